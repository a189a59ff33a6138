// GDN varlen chunked prefill for gfx950 (chunk C = 64, dk = dv = 128).
//
// A workgroup walks the chunks of one (sequence, v-head) chain, or of one slice
// of its state rows, as a two-stage pipeline:
//   * NP producer waves (NCW .. NCW+NP-1; four, or seven beside one consumer and six
//     beside two, which fill the workgroup's eight waves)
//     prepare chunk t: stage K and Q in LDS, form the gates, the masked/decayed
//     products N = strictLower(beta Gamma KK^T) and P = tril(Gamma QK^T), and
//     T~ = (I + N)^-1;
//   * the consumer waves (0 .. NCW-1) meanwhile advance the state through chunk t-1.
// Every LDS buffer a consumer reads (K, Q, T~, P, gates) is double-buffered by
// chunk parity (V is single-buffered and rewritten only after it was read).
// The roles hand chunks over through LDS counters, so each runs its own chain
// and neither waits for the other's sub-steps.  The fp32 state never leaves the
// register file: consumer wave w owns state rows v in [R0 + VW w, R0 + VW w + VW)
// as MFMA accumulators (16x16 tiles of S^T; lane = (k-group g = lane/16,
// column n = lane%16) holds S[v][k..k+3]).
//
// Launch variants (struct Variant): NCW consumer waves of VT 16-row tiles each
// cover ROWS = 16 NCW VT state rows, so F = 128 / ROWS workgroups share a chain,
// each owning rows [R0, R0 + ROWS).  They all prepare the same chunk data (the
// producer work does not depend on the state) and each stages only its slice of
// V.  Batches with many chains use F = 1 (four consumer waves of 32 rows); few
// chains are split so that every CU gets a workgroup (with F = 8 and F = 4 one or
// two 16-row consumers beside seven or six pipelined producers, since the chunk
// preparation, repeated in every slice, sets the pace).
//
// Batches of few chains can run in two kernels instead: a prep kernel prepares every
// chunk once (all chunks in parallel), and a state pass takes its T~, P and gates from
// memory.  Split 8 ways the state pass is gdn_prefill_state_kernel; split 4 or 2 ways it
// is a variant of the kernel above, whose loader waves copy the tiles where the producers
// would have computed them.  Split 4 and 8 ways the path runs in a caller's workspace or
// in the library's scratch, split 2 ways in the drop-in's scratch only (dropin_route).
//
// Per chunk (positions >= clen are zero-padded: K = Q = V = 0, beta = 0 and
// log-gate 0, as kernel_prefill.cu:102-114, 125-132 pads them):
//   gamma = inclusive cumsum of the log gates, beta = sigmoid(b)   (a1, :101-122;
//           summed in fp64 and kept as an fp32 pair, in log2 units)
//   N[i][j] = beta_i e^{gamma_i - gamma_j} k_i.k_j   (i > j)       (:134-146, sign folded)
//   P[i][j] = e^{gamma_i - gamma_j} q_i.k_j          (j <= i)       (:165-185; stored times scale)
//   T~ = (I + N)^-1                                   (:148-163)
//   X  = K S^T                                        (retrieval from the chunk-start state)
//   Y  = beta (V - e^gamma X)
//   v_new = T~ Y          (= T~(beta V) - T~(beta e^gamma K) S^T = U - W S^T, :187-195, 236-271)
//   o  = scale (e^gamma Q S^T + P v_new)              (:216-234, 273-283)
//   S  = e^{gamma_last} S + (d v_new)^T K,  d_c = e^{gamma_last - gamma_c}   (:197-202, 286-293)
//
// T~ is built in three steps: each producer wave forms one diagonal 16x16 tile of
// N; one wave inverts the four diagonal blocks D_I = (I + N_II)^-1 by forward
// substitution (16 lanes per block, one lane per column); two waves then form the
// off-diagonal blocks as a 2x2 block inverse over the 32x32 halves on 16x16x16
// MFMAs (offdiag_right / offdiag_left).
//
// Precision: q/k/v are exact bf16 MFMA operands.  Operands that are fp32 values
// (S, Y, N, T~, d*v_new) are split into bf16 hi + lo pairs so that the products
// feeding the state carry ~16 mantissa bits; fp32 accumulation throughout.  The
// output-only products (Q S^T and P v_new) use bf16 hi parts alone.  The residual
// x - hi(x) of a split is formed exactly on the matrix pipe (residual4).
//
// MFMA operand convention (v_mfma_f32_16x16x32_bf16): lane l supplies row/col
// l%16 and 8 contraction elements chosen by g = l/16.  A and B are paired with
// contraction index kappa(g, s) = 4g + s (s < 4), 16 + 4g + (s - 4) (s >= 4)
// inside each 32-wide block -- exactly what two 16x16 accumulator tiles stacked
// along the contraction dim hold, so accumulators become A or B operands without
// leaving registers.  LDS tiles keep their contraction columns in that order
// (perm32) so an operand row is one 16-byte read; an operand column of a
// row-major tile is two ds_read_b64_tr_b16 (transpose reads within 16 lanes).
#include <hip/hip_ext.h>

#include <atomic>
#include <mutex>
#include <thread>
#include <type_traits>

#include "gdn_common.hpp"
#include "gdn_launch.hpp"

namespace gdn {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

constexpr int C = 64;        // chunk length
constexpr int D = kHeadDim;  // 128
constexpr int KSTR = 128;    // bf16 row stride of the K and Q tiles (16-byte slots XOR-swizzled by row)
constexpr int VSTR = 144;    // bf16 row stride of the V tile (rows 32 bytes apart modulo 128)
constexpr int TSTR = 72;     // bf16 row stride of 64-wide tiles (T~, P, N)
constexpr int NDB = 16 * 16 + 4;  // floats per diagonal N block (column-major; padded by 16 bytes)
constexpr int NROWS = C - 16;  // rows of N kept for the off-diagonal solve

template <int NCW_, int VT_, bool HOOKS_ = false, bool LOAD_ = false, int NP_ = 4, bool PERSIST_ = false>
struct Variant {
  static constexpr bool kHooks = HOOKS_;         // testing hooks of PrefillArgs compiled in
  static constexpr bool kLoad = LOAD_;           // waves NCW.. load prepared T~/P (two-kernel path)
  static constexpr int NCW = NCW_;               // consumer waves
  static constexpr int NP = NP_;                 // producer (or loader) waves: 4; or 7 (6) beside one (two) consumers
  static constexpr int VT = VT_;                 // 16-row state tiles per consumer wave
  static constexpr int VW = 16 * VT;             // state rows per consumer wave
  static constexpr int ROWS = NCW * VW;          // state rows per workgroup
  static constexpr int F = 128 / ROWS;           // workgroups per chain
  static constexpr int NTHREADS = 64 * (NCW + NP);
  static constexpr int VSEG = 8 * ROWS;          // 16-byte segments of the V slice of a chunk
  // Seven producers beside one consumer, or six beside two, run pipelined one chunk
  // deep (producer_loop_split) with NP - 3 stager waves, and hand a chunk to the
  // consumers in two steps (K, Q, the gates and V; then T~ and P).
  static constexpr bool kPipelined = NP_ >= 6;
  static constexpr int kStagers = NP_ - 3;
  static_assert(F * ROWS == 128 && NCW + NP <= 8, "unsupported launch variant");
  static_assert(NP == 4 || (!LOAD_ && NCW + NP == 8 && NCW <= 2), "pipelined producers fill the workgroup");
  // One workgroup per CU runs a list of whole chains back to back
  // (gdn_prefill_persistent_kernel); the four-producer F = 1 layout only.
  static constexpr bool kPersist = PERSIST_;
  static_assert(!PERSIST_ || (NCW_ == 4 && VT_ == 2 && NP_ == 4 && !LOAD_), "persistent: F = 1 only");
};

// Production launch variants by split factor F (workgroups per chain).  With F = 8
// (F = 4) a chain's slice has one (two) 16-row consumer waves and the chunk
// preparation, repeated in every slice, sets the pace: seven (six) pipelined
// producer waves share it.
template <bool HOOKS>
using SplitVariant1 = Variant<4, 2, HOOKS>;
template <bool HOOKS>
using SplitVariant2 = Variant<4, 1, HOOKS>;
template <bool HOOKS>
using SplitVariant4 = Variant<2, 1, HOOKS, false, 6>;
template <bool HOOKS>
using SplitVariant8 = Variant<1, 1, HOOKS, false, 7>;
// F = 1 as one workgroup per CU running lists of chains (batches of many chains).
template <bool HOOKS>
using PersistVariant = Variant<4, 2, HOOKS, false, 4, true>;

// Prepared tiles of one chunk-head in the workspace (its image), in 16-byte units: the
// operand fragments of T~ hi, T~ lo and P that the state pass reads, in that order, six
// fragments each (tile_frag) of one unit per lane, so that an image is copied and its
// fragments are read linearly; then the chunk's gates beta_c, e^{gamma_c} and
// e^{gamma_last - gamma_c} (fp32, 64 each).  The strictly-upper blocks of fragments
// (0, 0) and (2, 1) are zeros.  The chunks of a batch (of the window of it that a launch
// covers) are numbered through, sequence after sequence (chunk_slots); chunk-head
// (slot n, v-head h) is image n Hv + h.
constexpr int kTileFrags = 6;
constexpr int kTileUnits1 = kTileFrags * 64;  // units of one tile
constexpr int kTileUnits = 3 * kTileUnits1;
constexpr int kGateUnits = 3 * C / 4;
constexpr int kTileImage = kTileUnits + kGateUnits;

// Fragment of a lower-triangular tile for rows 16 ct .. +15, contraction block js.
__device__ __forceinline__ constexpr int tile_frag(int ct, int js) { return ct < 2 ? ct : 2 * ct - 2 + js; }

constexpr int kMaxSortedSeqs = 1024;  // longest-first ordering up to this many sequences
constexpr int kMaxPersistList = 128;  // chains per workgroup of the persistent kernel
constexpr int kMaxPersistLpt = 64;    // batches of at most this many sequences get a longest-processing-time list

struct __align__(16) PrefillSmem {
  uint16_t K[2][C * KSTR];    // K chunk [c][perm(k)], by chunk parity
  uint16_t Q[2][C * KSTR];    // Q chunk [c][perm(k)]
  uint16_t Th[2][C * TSTR];   // T~ hi [c][perm(j)] (strictly-upper blocks stay 0)
  uint16_t Tl[2][C * TSTR];   // T~ lo
  uint16_t P[2][C * TSTR];    // P (bf16) [c][perm(j)] (strictly-upper blocks stay 0)
  uint16_t V[C * VSTR];       // V chunk [c][v], single-buffered (written after its last read)
  uint16_t Nh[NROWS * TSTR];  // N rows 16..63, hi [i - 16][perm(j)] (producers only; row block 0
  uint16_t Nl[NROWS * TSTR];  // of N is never an operand), lo
  float Nd[4 * NDB];          // diagonal 16x16 blocks of N (fp32, column-major: [block][col][row])
  float gam[2][C];            // gamma_c log2(e) (inclusive cumsum of the log2 gates), rounded
  float gaml[2][C];           // its rounding error (the sum is formed in fp64)
  float bet[2][C];            // beta_c
  float eg[2][C];             // e^{gamma_c}
  float dd[2][C];             // e^{gamma_last - gamma_c}
  int seq;                    // sequence handled by this workgroup
  int pseq[kMaxPersistList];  // persistent kernel: the sequences of the workgroup's chains, in order,
  int ps0[kMaxPersistList];   // their token ranges [ps0, ps1),
  int ps1[kMaxPersistList];
  int pcount;                 // and their number
  int plen[kMaxPersistLpt];   // persistent kernel, up to kMaxPersistLpt sequences: their lengths,
  int pstart[kMaxPersistLpt];  // starts and longest-first order (the list is formed while the
  int porder[kMaxPersistLpt];  // first chain runs)
  int sync[16];               // hand-off counters (enum SyncCounter)
  int spin_limit;             // kernels with testing hooks: polls before a hand-off wait gives up
  unsigned* aborts;           // kernels with testing hooks: optional count of waits that gave up
};

// Before a workgroup's first chunk its LDS tiles double as integer scratch: the
// longest-first ranking (pick_sequence) keeps up to kMaxSortedSeqs lengths in Nh, and
// the persistent kernel's boustrophedon lists keep lengths, starts and order of up to
// kMaxSortedSeqs sequences in V.
static_assert(kMaxSortedSeqs * sizeof(int) <= sizeof(PrefillSmem::Nh), "sequence lengths fit Nh");
static_assert(3 * kMaxSortedSeqs * sizeof(int) <= sizeof(PrefillSmem::V), "sequence lists fit V");

// LDS of one wave of the prep kernel (two-kernel path), where a wave prepares a whole
// chunk-head: what its lanes exchange.
struct __align__(16) PrepSmem {
  float gam[C];
  float gaml[C];
  float bet[C];
  uint16_t D[2][4 * 16 * 16];  // diagonal blocks of T~, hi and lo, column-major ([block][col][row])
  union {
    float Nd[4 * NDB];              // diagonal blocks of N (until they are inverted)
    uint16_t X[6][2][16 * 16];      // off-diagonal blocks of T~, hi and lo, column-major
  };
};
static_assert(12 * sizeof(PrepSmem) <= 160 * 1024, "three prep waves a SIMD");

// Gate arrays are copied from chunk images in 16-byte units, addressed from beta
// (gate_unit): 16-byte aligned, e^gamma and the update decay following it.
static_assert(offsetof(PrefillSmem, bet) % 16 == 0 &&
                  offsetof(PrefillSmem, eg) == offsetof(PrefillSmem, bet) + sizeof(PrefillSmem::bet) &&
                  offsetof(PrefillSmem, dd) == offsetof(PrefillSmem, eg) + sizeof(PrefillSmem::eg),
              "gate layout");

constexpr float kLog2e = 1.4426950408889634f;

// 2^{x} for x <= 0 (the hardware exp2, v_exp_f32).  Log gates are kept in log2
// units (gamma * log2(e)), so every decay e^{gamma_i - gamma_j} is one exp2.
__device__ __forceinline__ float exp2_le0(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ f32x4 mfma(const uint4& a, const uint4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                  __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }

// Raw buffer resource over [base, base + bytes): a vector store whose byte offset
// (plus its size) reaches past `bytes` is dropped by the hardware, which replaces a
// per-lane branch around stores that may fall outside a chunk.  The third dword is
// the gfx9 raw-buffer format word (32-bit data format, no swizzle, no stride).
typedef __amdgpu_buffer_rsrc_t BufferRsrc;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ BufferRsrc buffer_rsrc(void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(base, short(0), int(bytes), 0x00020000);
}
__device__ __forceinline__ void buffer_store16(u32x4 v, BufferRsrc r, int offset) {
  __builtin_amdgcn_raw_buffer_store_b128(v, r, offset, 0, 0);
}
__device__ __forceinline__ void buffer_store8(u32x2 v, BufferRsrc r, int offset) {
  __builtin_amdgcn_raw_buffer_store_b64(v, r, offset, 0, 0);
}

// Calls f(std::integral_constant<int, I>) for I = 0 .. N-1 (compile-time indices).
template <int I, int N, class Fn>
__device__ __forceinline__ void static_for_impl(Fn&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for_impl<I + 1, N>(f);
  }
}
template <int N, class Fn>
__device__ __forceinline__ void static_for(Fn&& f) {
  static_for_impl<0, N>(f);
}

// Position of contraction index r (0..31) inside a 32-wide permuted block.
__device__ __forceinline__ int perm32(int r) { return ((r & 15) >> 2) * 8 + ((r >> 4) << 2) + (r & 3); }
__device__ __forceinline__ int perm(int x) { return (x & ~31) + perm32(x & 31); }

// K/Q tiles: element (r, q) (q = permuted column) lives in 16-byte slot
// (q / 8) ^ sigma(r) of row r.  sigma swaps bits 1 and 2 of r (and keeps bits 0
// and 3): eight consecutive rows then hit eight different slots (row-operand
// reads are conflict-free), and the four rows of a transposed read split over
// two slot ranges.
__device__ __forceinline__ int kq_sigma(int r) { return (r & 9) | ((r & 2) << 1) | ((r & 4) >> 1); }
__device__ __forceinline__ int kq_off(int r, int q) { return r * KSTR + (((q >> 3) ^ kq_sigma(r)) << 3) + (q & 7); }

// Operand row of a K/Q tile: rows row0 + lane%16, contraction block ks.
__device__ __forceinline__ uint4 frag_kq(const uint16_t* tile, int row0, int ks, int lane) {
  return *reinterpret_cast<const uint4*>(tile + kq_off(row0 + (lane & 15), 32 * ks + 8 * (lane >> 4)));
}

// Operand row: rows row0 + lane%16, contraction block ks (32 wide), from a tile
// stored with permuted columns.
__device__ __forceinline__ uint4 frag(const uint16_t* tile, int stride, int row0, int ks, int lane) {
  return *reinterpret_cast<const uint4*>(tile + (row0 + (lane & 15)) * stride + 32 * ks + 8 * (lane >> 4));
}

// Operand row of a T~ or P tile, rows 16 ct + lane%16, contraction block js: from the
// producers' row-major tile, or (state pass) from the copied image's fragments.
template <bool kImage>
__device__ __forceinline__ uint4 tile_row(const uint16_t* tile, int ct, int js, int lane) {
  if constexpr (kImage) {
    return *reinterpret_cast<const uint4*>(tile + 8 * (64 * tile_frag(ct, js) + lane));
  } else {
    return frag(tile, TSTR, 16 * ct, js, lane);
  }
}

__device__ __forceinline__ uint2 read_tr(const uint16_t* p) {
  const i16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(p));
  return __builtin_bit_cast(uint2, v);
}

// Four rows k0 + 4g .. +3 of column col0 + lane%16 of a row-major tile whose
// columns are perm-ordered (groups of 4 columns stay contiguous).  In each
// 16-lane group, lane j reads 4 contiguous columns of row k0 + 4g + j/4; the
// transpose read hands lane i element i of each of those rows.
__device__ __forceinline__ uint2 col4_tr(const uint16_t* tile, int stride, int k0, int col0, int lane) {
  const int j = lane & 15, g = lane >> 4;
  return read_tr(tile + (k0 + 4 * g + (j >> 2)) * stride + perm(col0 + 4 * (j & 3)));
}


// Operand column of the K tile for the state update: column 16 kt + lane%16 (of
// the unpermuted k index), contraction rows 32 ks + kappa(g, s), as two
// transpose reads of 4 rows (k0 = 32 ks, then k0 + 16).  In 16-lane group g lane
// j reads 4 contiguous columns of row k0 + rl, rl = 4 g + j / 4, namely element
//   kq_off(k0 + rl, perm(16 kt + 4 (j & 3))),
// and perm(16 kt + 4 (j & 3)) = 32 (kt / 2) + 8 (j & 3) + 4 (kt & 1), so with
// s = sigma(rl) the offset is
//   (k0 + rl) KSTR + 32 ((kt / 2) ^ (s >> 2)) + 8 ((j & 3) ^ (s & 3)) + 4 (kt & 1):
// four lane bases (one per kt / 2) plus compile-time offsets.
struct KtBases {
  int b[4];
};
__device__ __forceinline__ KtBases kt_bases(int lane) {
  const int j = lane & 15, rl = 4 * (lane >> 4) + (j >> 2), sl = kq_sigma(rl);
  const int l0 = rl * KSTR + 8 * ((j & 3) ^ (sl & 3));
  KtBases r;
#pragma unroll
  for (int m = 0; m < 4; ++m) r.b[m] = l0 + 32 * (m ^ (sl >> 2));
  return r;
}
template <int KS, int KT>
__device__ __forceinline__ uint4 frag_tr_k_at(const uint16_t* tile, const KtBases& kb) {
  const uint16_t* p = tile + kb.b[KT / 2] + 32 * KS * KSTR + 4 * (KT & 1);
  const uint2 a = read_tr(p), b = read_tr(p + 16 * KSTR);
  return uint4{a.x, a.y, b.x, b.y};
}

// B/A operand (bf16 hi parts) from two accumulator tiles stacked along the
// contraction dim.
__device__ __forceinline__ uint4 pack_hi(const f32x4& t0, const f32x4& t1) {
  return uint4{pack_bf16x2(t0[0], t0[1]), pack_bf16x2(t0[2], t0[3]), pack_bf16x2(t1[0], t1[1]),
               pack_bf16x2(t1[2], t1[3])};
}

// 16x16x16 MFMA (one 16-wide contraction block): lane l supplies A[l%16][4g..4g+3]
// and B[4g..4g+3][l%16], g = l/16 -- the lower half of the 32-wide convention.
__device__ __forceinline__ f32x4 mfma16(const uint2& a, const uint2& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, a), __builtin_bit_cast(i16x4, b), c, 0,
                                                   0, 0);
}

// The residuals t - hi(t) of four fp32 values per lane, given their bf16 hi parts
// packed as a 16x16x16 B operand (lane l, slot s: B[4g + s][l%16]), formed on the
// matrix pipe: D = t + (-I) hi(t) with t as the accumulator, which lane l holds as
// D[4g + s][l%16] -- the same (lane, slot) for every element, so this is an
// elementwise t - hi(t).  Each element has one nonzero product and its exact result
// is representable, so the residual is exact (as the fp32 subtraction would be),
// and the wave issues one MFMA instead of eight VALU instructions.  -I as the A
// operand (lane l: row l%16, contraction 4g + s) has its one nonzero, bf16 -1, in
// slot l%4 when g == (l%16)/4.
__device__ __forceinline__ f32x4 residual4(const f32x4& t, const uint2& hi) {
  const uint32_t l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const uint32_t w = (l >> 4) == ((l & 15) >> 2) ? (0xbf80u << (16 * (l & 1))) : 0u;
  const uint2 neg_identity = (l & 2) ? uint2{0u, w} : uint2{w, 0u};
  return mfma16(neg_identity, hi, t);
}

// bf16 hi parts (round to nearest even) and lo parts (the residual, rounded) of
// two stacked accumulator tiles (B/A operands, as pack_hi) or of one.
__device__ __forceinline__ void split_pack(const f32x4& t0, const f32x4& t1, uint4& hi, uint4& lo) {
  hi = pack_hi(t0, t1);
  const f32x4 r0 = residual4(t0, uint2{hi.x, hi.y}), r1 = residual4(t1, uint2{hi.z, hi.w});
  lo = uint4{pack_bf16x2(r0[0], r0[1]), pack_bf16x2(r0[2], r0[3]), pack_bf16x2(r1[0], r1[1]),
             pack_bf16x2(r1[2], r1[3])};
}
__device__ __forceinline__ void split4(const f32x4& t, uint2& hi, uint2& lo) {
  hi = uint2{pack_bf16x2(t[0], t[1]), pack_bf16x2(t[2], t[3])};
  const f32x4 r = residual4(t, hi);
  lo = uint2{pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3])};
}

__device__ __forceinline__ int64_t load_cu(const void* cu, int is64, int i) {
  return is64 ? static_cast<const int64_t*>(cu)[i] : int64_t(static_cast<const int32_t*>(cu)[i]);
}

// Tokens [s0, s1) of sequence i, its offsets clamped into [0, T]; two-kernel path: of the
// launch's window of it (win_tokens tokens from win_begin on; 0 = the whole sequence).
struct SeqRange {
  int64_t s0, s1;
};
__device__ __forceinline__ SeqRange seq_range(const PrefillArgs& p, int i) {
  int64_t a = load_cu(p.cu_seqlens, p.cu_is_64, i), b = load_cu(p.cu_seqlens, p.cu_is_64, i + 1);
  a = a < 0 ? 0 : (a > p.T ? p.T : a);
  b = b < a ? a : (b > p.T ? p.T : b);
  if (p.win_tokens > 0) {
    a += p.win_begin;
    a = a < b ? a : b;
    b = b - a < p.win_tokens ? b : a + p.win_tokens;
  }
  return SeqRange{a, b};
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int dpp_or_zero(int x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, ROW_MASK, 0xF, true);
}

// Inclusive prefix sum of an int over the wavefront (the DPP steps of
// wave_inclusive_scan2).
__device__ __forceinline__ int wave_inclusive_scan(int x) {
  x += dpp_or_zero<0x111, 0xF>(x);
  x += dpp_or_zero<0x112, 0xF>(x);
  x += dpp_or_zero<0x114, 0xF>(x);
  x += dpp_or_zero<0x118, 0xF>(x);
  x += dpp_or_zero<0x142, 0xA>(x);
  x += dpp_or_zero<0x143, 0xC>(x);
  return x;
}

// Chunks of the sequences before sequence `seq` (a wave-uniform call of a whole wave):
// the number of its first chunk among the batch's chunk images.  With valid offsets the
// batch has at most T / C + N chunks, with any at most N ceil(T / C).
__device__ int chunks_before(const PrefillArgs& p, int seq, int lane) {
  int before = 0;
  for (int base = 0; base < seq; base += 64) {
    int n = 0;
    if (base + lane < seq) {
      const SeqRange r = seq_range(p, base + lane);
      n = int((r.s1 - r.s0 + C - 1) / C);
    }
    before += __builtin_amdgcn_readlane(wave_inclusive_scan(n), 63);
  }
  return before;
}

// Chunk number `slot` of the batch: its first token and its length (0 if the batch has
// fewer chunks), and the batch's number of chunks; wave-uniform.  (Token indices fit 31
// bits.)
struct ChunkAt {
  int start, clen, total;
};
__device__ __forceinline__ ChunkAt find_chunk(const PrefillArgs& p, int slot, int lane) {
  if (p.N == 1) {
    const SeqRange r = seq_range(p, 0);
    const int64_t cs = r.s0 + int64_t(slot) * C;
    return ChunkAt{int(cs), cs >= r.s1 ? 0 : int(r.s1 - cs < C ? r.s1 - cs : C), int((r.s1 - r.s0 + C - 1) / C)};
  }
  ChunkAt c = {0, 0, 0};
  for (int base = 0; base < p.N; base += 64) {
    SeqRange r = {0, 0};
    if (base + lane < p.N) r = seq_range(p, base + lane);
    const int n = int((r.s1 - r.s0 + C - 1) / C);
    const int end = wave_inclusive_scan(n) + c.total;
    const uint64_t hit = __builtin_amdgcn_ballot_w64(slot >= end - n && slot < end);
    if (hit != 0) {
      const int l = __builtin_ctzll(hit);
      c.start = __builtin_amdgcn_readlane(int(r.s0), l) + C * (slot - __builtin_amdgcn_readlane(end - n, l));
      c.clen = min(__builtin_amdgcn_readlane(int(r.s1), l) - c.start, C);
    }
    c.total = __builtin_amdgcn_readlane(end, 63);
  }
  return c;
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_or_zero_f64(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, uint32_t(u), CTRL, ROW_MASK, 0xF, true);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, uint32_t(u >> 32), CTRL, ROW_MASK, 0xF, true);
  return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}

// Inclusive prefix sum over the 64 lanes of a wavefront with DPP: shifts by
// 1, 2, 4, 8 inside each 16-lane row, then lane 15 of rows 0 / 2 into rows 1 / 3
// (row_bcast:15) and lane 31 into rows 2 and 3 (row_bcast:31).  The sum runs in
// fp64 and is returned as a pair hi + lo of floats (lo = the rounding error of
// hi): the decays e^{gamma_i - gamma_j} are formed from differences of these
// sums, and with fast decay the sums reach 1e5 in magnitude while a difference
// that matters (one that does not underflow to zero) is below 1e2 -- a plain
// fp32 difference would carry the sums' rounding error, up to about 1e-2.
__device__ __forceinline__ float wave_inclusive_scan2(float x, float& lo) {
  double d = x;
  d += dpp_or_zero_f64<0x111, 0xF>(d);
  d += dpp_or_zero_f64<0x112, 0xF>(d);
  d += dpp_or_zero_f64<0x114, 0xF>(d);
  d += dpp_or_zero_f64<0x118, 0xF>(d);
  d += dpp_or_zero_f64<0x142, 0xA>(d);
  d += dpp_or_zero_f64<0x143, 0xC>(d);
  const float hi = float(d);
  lo = float(d - double(hi));
  return hi;
}

// gamma_i - gamma_j from the pairs (hi, lo) of the compensated scan.  The hi
// difference is exact whenever it is small against the sums (Sterbenz), so the
// result is accurate to fp32 precision of the difference itself.
__device__ __forceinline__ float gamma_diff(float hi_i, float lo_i, float hi_j, float lo_j) {
  return (hi_i - hi_j) + (lo_i - lo_j);
}

// Log-space decay in log2 units, -exp(A_log) * softplus(a + dt_bias) * log2(e)
// (torch threshold 20), with the hardware exp2/log2; neg_decay = -exp(A_log).
// log2(1 + 2^y) is softplus(x) * log2(e) with y = x log2(e), so no conversion
// back to natural units is needed.  For very negative arguments log2(1 + 2^y)
// loses its relative accuracy but stays within ~2e-7 absolutely.
__device__ __forceinline__ float fast_log2_gate(float neg_decay, float x) {
  const float y = x * kLog2e;
  return neg_decay * (x > 20.f ? y : __builtin_amdgcn_logf(1.f + __builtin_amdgcn_exp2f(y)));
}

__device__ __forceinline__ float fast_sigmoid(float x) {
  return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-x * 1.4426950408889634f));
}

// Orders this wave's LDS writes before its later LDS reads by other lanes.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace

// Waves on this device whose hand-off wait gave up (see wait_count), since the
// library was loaded or the count was last reset; read by prefill_giveups.
__device__ unsigned int gdn_prefill_giveup_count;

namespace {

// Hand-off between the two roles: monotonically increasing LDS counters.  A wave
// signals by adding 1 after its earlier LDS accesses (release: see signal_count); a
// waiter polls until the count reaches its target (acquire).
enum SyncCounter {
  kReady = 0,     // chunk handed over to the consumers (4 a chunk; pipelined: its T~ and P, NS + 2)
  kVFree = 1,     // consumers read the chunk's V
  kConsumed = 2,  // consumers done with the chunk's buffers
  kPPhase = 3,    // four producers: their step barriers; pipelined: solve and N tiles done (3 a chunk)
  kAbort = 4,     // a wait gave up
  kDiagN = 5,     // diagonal N tiles formed (4 a chunk)
  kX32 = 6,       // off-diagonal block X32 stored
  kStaged = 7,    // pipelined: the chunk's K/Q staged and its gates stored (NS + 1 a chunk)
  kNRead = 8,     // pipelined: the left off-diagonal wave read its N operands
  kVStaged = 9,   // pipelined: the chunk's V staged (NS a chunk)
  kList = 10      // persistent kernel: the workgroup's chain list is complete (1)
};
constexpr int kSpinLimit = 1 << 21;  // default polls (about 70 ms) before a wait gives up

// Every hand-off publishes LDS data (or releases LDS reads) to waves of the same
// workgroup, through an LDS counter.  The LDS performs a CU's operations in one
// order, and a wave's own LDS operations in the order the wave issues them, so the
// increment is performed after every LDS write or read the wave issued before it,
// and a waiter that sees the count issues its reads after that.  No wait for the
// wave's outstanding LDS operations is needed before the increment (a workgroup-
// scope release fence would add one, s_waitcnt lgkmcnt(0), which stalls the
// signalling wave until its last writes land); the compiler-level fences keep the
// program order.  Nothing is published through these counters in global memory.
template <class Smem>
__device__ __forceinline__ void signal_count(Smem& sm, int which, int lane) {
  (void)lane;
  // One LDS add from lane 0, with exec set to that lane inside one asm block rather
  // than by a branch, so that the surrounding arithmetic is still scheduled as one
  // block.  Every caller runs with the whole wave active.  The block writes no SCC
  // (s_mov only), and the compiler does not count its LDS operation in its waits, which
  // can only make those stricter (a wave's LDS operations complete in order).
  typedef __attribute__((address_space(3))) int lds_int;
  const uint32_t addr = uint32_t(reinterpret_cast<uintptr_t>((lds_int*)(&sm.sync[which])));
  uint64_t saved;
  asm volatile(
      "s_mov_b64 %0, exec\n\t"
      "s_mov_b64 exec, 1\n\t"
      "ds_add_u32 %1, %2\n\t"
      "s_mov_b64 exec, %0"
      : "=&s"(saved)
      : "v"(addr), "v"(1)
      : "memory");
}

// Waits until counter `which` reaches `target`.  Every wait is bounded: if one
// ever gives up (which only a logic error, or the testing hooks of PrefillArgs,
// can cause), it raises kAbort, and all later waits return at once, so the
// workgroup still finishes instead of hanging.  The wave that gives up adds 1 to
// gdn_prefill_giveup_count (a global atomic from one lane), and the workgroup
// writes NaN to every output element and state element it owns, so wrong results never
// look valid.  Production kernels give up after kSpinLimit polls; kernels built with the
// hooks after sm.spin_limit polls, also counting each give-up in sm.aborts if set.
template <bool kHooks, class Smem>
__device__ __forceinline__ void wait_count(Smem& sm, int which, int target) {
  if (__hip_atomic_load(&sm.sync[which], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < target) {
    for (int it = 0;; ++it) {
      __builtin_amdgcn_s_sleep(1);
      if (__hip_atomic_load(&sm.sync[which], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= target) break;
      if (__hip_atomic_load(&sm.sync[kAbort], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0) break;
      int limit = kSpinLimit;
      if constexpr (kHooks) limit = sm.spin_limit;
      if (it >= limit) {
        __hip_atomic_store(&sm.sync[kAbort], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) == 0) {
          __hip_atomic_fetch_add(&gdn_prefill_giveup_count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if constexpr (kHooks) {
            unsigned* aborts = sm.aborts;
            if (aborts) __hip_atomic_fetch_add(aborts, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
        break;
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// wait_count for counter `a`, reading counter `b` in the same LDS round trip:
// returns whether `b` had reached `tb` then, so that a later wait for it can be
// skipped (the acquire that ends this wait covers both).
template <bool kHooks, class Smem>
__device__ __forceinline__ bool wait_count_peek(Smem& sm, int a, int ta, int b, int tb) {
  const int va = __hip_atomic_load(&sm.sync[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  const int vb = __hip_atomic_load(&sm.sync[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  const bool b_ok = __builtin_amdgcn_readfirstlane(int(vb >= tb)) != 0;
  if (__builtin_amdgcn_readfirstlane(int(va >= ta)) != 0) {
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  } else {
    wait_count<kHooks>(sm, a, ta);
  }
  return b_ok;
}

template <class Smem>
__device__ __forceinline__ bool aborted(Smem& sm) {
  return __hip_atomic_load(&sm.sync[kAbort], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0;
}

constexpr uint32_t kNaNx2 = 0x7fc07fc0u;  // two bf16 quiet NaNs


// The parity-selected LDS buffers of one chunk.
struct ChunkBufs {
  uint16_t* K;
  uint16_t* Q;
  uint16_t* Th;
  uint16_t* Tl;
  uint16_t* P;
  float* gam;
  float* gaml;
  float* bet;
  float* eg;
  float* dd;
};

template <class Smem>
__device__ __forceinline__ ChunkBufs chunk_bufs(Smem& sm, int b) {
  return ChunkBufs{sm.K[b],   sm.Q[b],   sm.Th[b],  sm.Tl[b], sm.P[b],
                   sm.gam[b], sm.gaml[b], sm.bet[b], sm.eg[b], sm.dd[b]};
}

// ---------------------------------------------------------------------------
// Producer side (waves NCW .. NCW+3)
// ---------------------------------------------------------------------------

// Tiles of N and P from the staged K and Q (16x16 tiles, 4 MFMAs each).
//   kind 1: off-diagonal block (I, J), I > J, of N (bf16 hi/lo), from tile
//           K_J K_I^T so that a lane holds 4 consecutive columns of one row
//   kind 2: block (I, J), J <= I, of P, from tile K_J Q_I^T
struct TileJob {
  int kind, I, J;
};

__device__ __forceinline__ f32x4 ld4(const float* p) {
  const float4 x = *reinterpret_cast<const float4*>(p);
  return f32x4{x.x, x.y, x.z, x.w};
}

// Branch-free epilogues: gamma is non-increasing along the chunk, so every
// exponent kept is <= 0; the masked ones are clamped to 0 before the select.
template <class Smem>
__device__ __forceinline__ void tile_epilogue(Smem& sm, const ChunkBufs& cb, const TileJob t, const f32x4& acc,
                                              float scale, int lane) {
  const int g = lane >> 4, n16 = lane & 15;
  if (t.kind == 1) {
    // acc[i] = k_c . k_r, c = 16J + 4g + i, r = 16I + n16  ->  N[r][c]  (r > c)
    const int r = 16 * t.I + n16;
    const float gr = cb.gam[r], grl = cb.gaml[r], br = cb.bet[r];
    const f32x4 gcv = ld4(cb.gam + 16 * t.J + 4 * g), gcl = ld4(cb.gaml + 16 * t.J + 4 * g);
    f32x4 x;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = br * exp2_le0(fminf(gamma_diff(gr, grl, gcv[i], gcl[i]), 0.f)) * acc[i];
    uint2 hi, lo;
    split4(x, hi, lo);
    const int pos = (r - 16) * TSTR + perm(16 * t.J + 4 * g);
    *reinterpret_cast<uint2*>(sm.Nh + pos) = hi;
    *reinterpret_cast<uint2*>(sm.Nl + pos) = lo;
  } else {
    // acc[i] = k_j . q_c, j = 16J + 4g + i, c = 16I + n16  ->  P[c][j]  (j <= c),
    // with the output scale folded in
    const int c = 16 * t.I + n16;
    const float gc = cb.gam[c], gcl = cb.gaml[c];
    const f32x4 gj = ld4(cb.gam + 16 * t.J + 4 * g), gjl = ld4(cb.gaml + 16 * t.J + 4 * g);
    float pv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = exp2_le0(fminf(gamma_diff(gc, gcl, gj[i], gjl[i]), 0.f)) * (acc[i] * scale);
      pv[i] = 16 * t.J + 4 * g + i <= c ? x : 0.f;
    }
    *reinterpret_cast<uint2*>(cb.P + c * TSTR + perm(16 * t.J + 4 * g)) =
        uint2{pack_bf16x2(pv[0], pv[1]), pack_bf16x2(pv[2], pv[3])};
  }
}

template <int NJ, class Smem>
__device__ __forceinline__ void run_tiles(Smem& sm, const ChunkBufs& cb, const TileJob (&jobs)[NJ], float scale,
                                          int lane) {
  f32x4 acc[NJ];
#pragma unroll
  for (int t = 0; t < NJ; ++t) acc[t] = zero4();
  uint4 a[NJ][4], b[NJ][4];  // all operands first: one round of LDS latency
#pragma unroll
  for (int t = 0; t < NJ; ++t) {
    const TileJob j = jobs[t];
    const int arow = 16 * j.J;
    const uint16_t* btile = j.kind == 2 ? cb.Q : cb.K;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      a[t][ks] = frag_kq(cb.K, arow, ks, lane);
      b[t][ks] = frag_kq(btile, 16 * j.I, ks, lane);
    }
  }
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int t = 0; t < NJ; ++t) acc[t] = mfma(a[t][ks], b[t][ks], acc[t]);
#pragma unroll
  for (int t = 0; t < NJ; ++t) tile_epilogue(sm, cb, jobs[t], acc[t], scale, lane);
}

// The four diagonal blocks of T~, D_I = (I + N_II)^-1.  diag_tiles forms N_II
// from the tiles K_I K_I^T (scaled as in the off-diagonal epilogue) for blocks
// I0 .. I1-1, stored column-major; diag_solve (one wavefront, all four blocks;
// diag_columns) then has lane (r, j) = (lane/16, lane%16) invert block r, column j,
// x = D_r[:, j], by right-looking forward substitution:
//   x_m = delta_mj - a_m,  a_i += N[i][m] x_m  for i > m
// (for m < j every term is zero, so x_m = 0 there).  The column of N needed at
// step m is one broadcast read per four rows; no cross-lane traffic.
template <int I0, int I1, class Smem>
__device__ __forceinline__ void diag_tiles(Smem& sm, const ChunkBufs& cb, int lane) {
  const int g = lane >> 4, n16 = lane & 15;
  {
    f32x4 acc[4];
#pragma unroll
    for (int I = I0; I < I1; ++I) {
      uint4 kf[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) kf[ks] = frag_kq(cb.K, 16 * I, ks, lane);
      acc[I] = zero4();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) acc[I] = mfma(kf[ks], kf[ks], acc[I]);
    }
    // acc[I][i] = k_r . k_c, r = 16I + 4g + i, c = 16I + n16 -> N[r][c] for r > c
    // (entries with r <= c are never read).
#pragma unroll
    for (int I = I0; I < I1; ++I) {
      const float gc = cb.gam[16 * I + n16], gcl = cb.gaml[16 * I + n16];
      const f32x4 gr = ld4(cb.gam + 16 * I + 4 * g), grl = ld4(cb.gaml + 16 * I + 4 * g);
      const f32x4 br = ld4(cb.bet + 16 * I + 4 * g);
      f32x4 x;
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = br[i] * exp2_le0(fminf(gamma_diff(gr[i], grl[i], gc, gcl), 0.f)) * acc[I][i];
      *reinterpret_cast<f32x4*>(sm.Nd + I * NDB + n16 * 16 + 4 * g) = x;
    }
  }
}

__device__ __forceinline__ void diag_columns(const float* Nd, float (&x)[16], int lane) {
  const int r = lane >> 4, j = lane & 15;
  const float* nb = Nd + r * NDB;
  // Columns are read kColAhead steps ahead of their use.
  constexpr int kColAhead = 4;
  f32x4 colv[15][4];
#pragma unroll
  for (int m = 0; m < kColAhead; ++m)
#pragma unroll
    for (int q = (m + 1) / 4; q < 4; ++q) colv[m][q] = ld4(nb + m * 16 + 4 * q);
  float a[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) {
    x[m] = (m == j) ? 1.f : (m == 0 ? 0.f : -a[m]);
    if (m + kColAhead < 15) {
#pragma unroll
      for (int q = (m + kColAhead + 1) / 4; q < 4; ++q)
        colv[m + kColAhead][q] = ld4(nb + (m + kColAhead) * 16 + 4 * q);
    }
    if (m < 15) {
#pragma unroll
      for (int q = (m + 1) / 4; q < 4; ++q) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 4 * q + e;
          if (i > m) a[i] = m == 0 ? colv[m][q][e] * x[0] : fmaf(colv[m][q][e], x[m], a[i]);
        }
      }
    }
  }
}

template <class Smem>
__device__ __forceinline__ void diag_solve(Smem& sm, const ChunkBufs& cb, int lane) {
  const int r = lane >> 4, j = lane & 15;
  float x[16];
  diag_columns(sm.Nd, x, lane);
  // rows 16r + i, column 16r + j of T~
  const int colp = perm(16 * r + j);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint2 hi, lo;
    split4(f32x4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]}, hi, lo);
    const uint32_t h4[4] = {hi.x, hi.x >> 16, hi.y, hi.y >> 16}, l4[4] = {lo.x, lo.x >> 16, lo.y, lo.y >> 16};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      cb.Th[(16 * r + 4 * q + e) * TSTR + colp] = uint16_t(h4[e]);
      cb.Tl[(16 * r + 4 * q + e) * TSTR + colp] = uint16_t(l4[e]);
    }
  }
}

struct Pair2 {  // bf16 hi / lo parts of a 16x16x16 operand
  uint2 h, l;
};

// acc += A B, both as hi/lo pairs (three passes).
__device__ __forceinline__ f32x4 mul3_16(f32x4 acc, const Pair2& a, const Pair2& b) {
  acc = mfma16(a.h, b.h, acc);
  acc = mfma16(a.h, b.l, acc);
  acc = mfma16(a.l, b.h, acc);
  return acc;
}

// B operand from an fp32 accumulator tile.
__device__ __forceinline__ Pair2 acc_b(const f32x4& t) {
  Pair2 r;
  split4(t, r.h, r.l);
  return r;
}

// A operand of the 16x16 block (I, J) of a hi/lo tile pair with permuted columns
// (row0 = first row held by the tiles).
__device__ __forceinline__ Pair2 block_a(const uint16_t* th, const uint16_t* tl, int row0, int I, int J, int lane) {
  const int off = (16 * I - row0 + (lane & 15)) * TSTR + perm(16 * J + 4 * (lane >> 4));
  return Pair2{*reinterpret_cast<const uint2*>(th + off), *reinterpret_cast<const uint2*>(tl + off)};
}

// B operand of the diagonal block D_J of T~.
__device__ __forceinline__ Pair2 diag_b(const ChunkBufs& cb, int J, int lane) {
  return Pair2{col4_tr(cb.Th, TSTR, 16 * J, 16 * J, lane), col4_tr(cb.Tl, TSTR, 16 * J, 16 * J, lane)};
}

// Writes an off-diagonal block X_IJ (accumulator layout) to Th/Tl.
__device__ __forceinline__ void store_block(const ChunkBufs& cb, const f32x4& X, int I, int J, int lane) {
  const int g = lane >> 4, col = perm(16 * J + (lane & 15));
  uint2 hi, lo;
  split4(X, hi, lo);
  const uint32_t h4[4] = {hi.x, hi.x >> 16, hi.y, hi.y >> 16}, l4[4] = {lo.x, lo.x >> 16, lo.y, lo.y >> 16};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    cb.Th[(16 * I + 4 * g + i) * TSTR + col] = uint16_t(h4[i]);
    cb.Tl[(16 * I + 4 * g + i) * TSTR + col] = uint16_t(l4[i]);
  }
}

// X_IJ = D_I (-G): written to Th/Tl and returned.
__device__ __forceinline__ f32x4 finish_block(const ChunkBufs& cb, const f32x4& G, const Pair2& dI, int I, int J,
                                              int lane) {
  const f32x4 X = mul3_16(zero4(), dI, acc_b(-G));
  store_block(cb, X, I, J, lane);
  return X;
}

// Off-diagonal blocks of T~, as a 2x2 block inverse over the 32x32 halves:
//   T~ = [[A^-1, 0], [-B^-1 C A^-1, B^-1]] with
//   A^-1 = [[D0, 0], [X10, D1]],  B^-1 = [[D2, 0], [X32, D3]],  C = [[N20, N21], [N30, N31]],
//   X10 = -D1 N10 D0,  X32 = -D3 N32 D2,  M = C A^-1,  [[X20, X21], [X30, X31]] = -B^-1 M.
// Two wavefronts share it.  Column 1 of M (N21 D1, N31 D1) does not need X10,
// so one wave forms X32, X21 and X31 (offdiag_right) while the other forms X10,
// X20 and X30 (offdiag_left); the left wave reads X32 back from T~ once the
// right wave has stored it (counter kX32).  Each wave reads all of its LDS
// operands before its first block store.
template <class Smem>
__device__ __forceinline__ void offdiag_right(Smem& sm, const ChunkBufs& cb, int t, int lane) {
  const Pair2 d1 = diag_b(cb, 1, lane), d2 = diag_b(cb, 2, lane);
  const Pair2 a2 = block_a(cb.Th, cb.Tl, 0, 2, 2, lane), a3 = block_a(cb.Th, cb.Tl, 0, 3, 3, lane);
  const Pair2 n21 = block_a(sm.Nh, sm.Nl, 16, 2, 1, lane), n31 = block_a(sm.Nh, sm.Nl, 16, 3, 1, lane),
              n32 = block_a(sm.Nh, sm.Nl, 16, 3, 2, lane);
  const f32x4 g32 = mul3_16(zero4(), n32, d2);
  const f32x4 m21 = mul3_16(zero4(), n21, d1);
  const f32x4 m31 = mul3_16(zero4(), n31, d1);
  finish_block(cb, g32, a3, 3, 2, lane);  // X32
  signal_count(sm, kX32, lane);
  const Pair2 x32t = acc_b(mul3_16(zero4(), acc_b(-g32), a3));  // A operand holding X32
  const Pair2 nm21 = acc_b(-m21), nm31 = acc_b(-m31);
  store_block(cb, mul3_16(zero4(), a2, nm21), 2, 1, lane);                           // X21
  store_block(cb, mul3_16(mul3_16(zero4(), x32t, nm21), a3, nm31), 3, 1, lane);      // X31
  (void)t;
}

template <bool kHooks, bool kSignalNRead = false, class Smem>
__device__ __forceinline__ void offdiag_left(Smem& sm, const ChunkBufs& cb, int t, int lane) {
  const Pair2 d0 = diag_b(cb, 0, lane);
  const Pair2 a1 = block_a(cb.Th, cb.Tl, 0, 1, 1, lane), a2 = block_a(cb.Th, cb.Tl, 0, 2, 2, lane),
              a3 = block_a(cb.Th, cb.Tl, 0, 3, 3, lane);
  const Pair2 n10 = block_a(sm.Nh, sm.Nl, 16, 1, 0, lane), n20 = block_a(sm.Nh, sm.Nl, 16, 2, 0, lane),
              n21 = block_a(sm.Nh, sm.Nl, 16, 2, 1, lane), n30 = block_a(sm.Nh, sm.Nl, 16, 3, 0, lane),
              n31 = block_a(sm.Nh, sm.Nl, 16, 3, 1, lane);
  // (Seven producers: the N tiles of the next chunk may be written once these reads
  // are done; the signal's release waits for them.)
  if constexpr (kSignalNRead) signal_count(sm, kNRead, lane);
  const f32x4 g10 = mul3_16(zero4(), n10, d0);
  const f32x4 p20 = mul3_16(zero4(), n20, d0);
  const f32x4 p30 = mul3_16(zero4(), n30, d0);
  const f32x4 x10 = finish_block(cb, g10, a1, 1, 0, lane);  // X10
  const Pair2 b10 = acc_b(x10);
  const Pair2 nm20 = acc_b(-mul3_16(p20, n21, b10));
  const Pair2 nm30 = acc_b(-mul3_16(p30, n31, b10));
  store_block(cb, mul3_16(zero4(), a2, nm20), 2, 0, lane);  // X20
  const f32x4 x30 = mul3_16(zero4(), a3, nm30);
  wait_count<kHooks>(sm, kX32, t + 1);  // X32 stored by the right wave
  const Pair2 x32 = block_a(cb.Th, cb.Tl, 0, 3, 2, lane);
  store_block(cb, mul3_16(x30, x32, nm20), 3, 0, lane);     // X30
}

// Global loads.  A CU streams about 48 KB of K, Q and V per chunk through its
// vector-memory pipe, and a wave that issues loads while that queue is full
// stalls until it drains.  The producers issue the next chunk's K/Q loads at
// the start of their middle step, while the consumers' retrieve (the heaviest
// LDS reader) runs, so the stall overlaps LDS work that would hold them up
// anyway.
//
// With NT threads sharing the K/Q rows of a chunk, thread pt (0..NT-1) owns K/Q
// segments pt + NT it: token pt/16 + (NT/16) it, columns 8 (pt%16) .. +7 (16
// consecutive threads read one 256-byte row); four producer waves (NT = 256) take
// tokens pt/16 + 16 it, it = 0..3.  Addresses are a wave-uniform chunk base (64-bit,
// scalar) plus a 32-bit lane offset that is fixed across chunks.
constexpr int NPROD = 256;  // producer threads (four waves)

template <int NT>
struct ProducerPrefetchT {
  static constexpr int RS = NT / 16;              // tokens between a thread's segments
  static constexpr int NIT = (C + RS - 1) / RS;   // segments per thread
  static_assert(NT % 64 == 0 && NT >= 64 && NT <= 256, "whole waves share the staging");
  uint4 k[NIT], q[NIT];
  uint16_t a, b;  // raw gate inputs of token pt (first wave only)
};
using ProducerPrefetch = ProducerPrefetchT<NPROD>;

struct LaneOffsets {
  int k, q;  // (pt/16) rows + 8 (pt%16) elements, in the K and Q row strides
  int ab;    // pt rows of the a/b [T, Hv] layout
};

template <int NT>
__device__ __forceinline__ void producer_prefetch(const PrefillArgs& p, int64_t cs, int clen, int h, int hq, int hk,
                                                  int pt, const LaneOffsets& lo, ProducerPrefetchT<NT>& f) {
  constexpr int RS = ProducerPrefetchT<NT>::RS;
  const uint16_t* kb = p.k + (cs * p.Hk + hk) * D;
  const uint16_t* qb = p.q + (cs * p.Hq + hq) * D;
#pragma unroll
  for (int it = 0; it < ProducerPrefetchT<NT>::NIT; ++it) {
    const int c = (pt >> 4) + RS * it;
    f.k[it] = f.q[it] = uint4{0u, 0u, 0u, 0u};
    if (c < clen) {
      f.k[it] = *reinterpret_cast<const uint4*>(kb + (lo.k + RS * it * p.Hk * D));
      f.q[it] = *reinterpret_cast<const uint4*>(qb + (lo.q + RS * it * p.Hq * D));
    }
  }
  if (pt < 64) {  // wave-uniform; the row index is clamped and padding masked when used
    const int off = pt < clen ? lo.ab : (clen - 1) * p.Hv;
    f.a = (p.a + cs * p.Hv + h)[off];
    f.b = (p.b + cs * p.Hv + h)[off];
  }
}

// The gates of token `lane` of a chunk (first producer wave, from the raw a/b
// values of its prefetch): the log2-gate prefix sum as an fp32 pair, beta,
// e^gamma and the update decay e^{gamma_last - gamma}.
struct ChunkGates {
  float gam, gaml, bet, eg, dd;
};

template <int NT>
__device__ __forceinline__ ChunkGates chunk_gates(const ProducerPrefetchT<NT>& f, int lane, int clen, float neg_decay,
                                                  float dt_bias) {
  const float lg = lane < clen ? fast_log2_gate(neg_decay, bf16_to_f32(f.a) + dt_bias) : 0.f;
  ChunkGates g;
  g.bet = lane < clen ? fast_sigmoid(bf16_to_f32(f.b)) : 0.f;
  g.gam = wave_inclusive_scan2(lg, g.gaml);
  const float glast = readlane_f(g.gam, clen - 1), glastl = readlane_f(g.gaml, clen - 1);
  g.eg = exp2_le0(g.gam);
  g.dd = exp2_le0(fminf(gamma_diff(glast, glastl, g.gam, g.gaml), 0.f));
  return g;
}

__device__ __forceinline__ void store_gates(const ChunkBufs& cb, const ChunkGates& g, int lane) {
  cb.gam[lane] = g.gam;
  cb.gaml[lane] = g.gaml;
  cb.bet[lane] = g.bet;
  cb.eg[lane] = g.eg;
  cb.dd[lane] = g.dd;
}

// Step 1 of a chunk: the prefetched K and Q rows into the chunk's tiles
// (permuted columns).
template <int NT>
__device__ __forceinline__ void stage_kq(const ChunkBufs& cb, const ProducerPrefetchT<NT>& f, int pt) {
  constexpr int RS = ProducerPrefetchT<NT>::RS;
#pragma unroll
  for (int it = 0; it < ProducerPrefetchT<NT>::NIT; ++it) {
    const int c = (pt >> 4) + RS * it, sg = pt & 15;
    if (RS * ProducerPrefetchT<NT>::NIT > C && c >= C) break;  // past the chunk (NT not dividing 1024)
    const int col0 = (8 * sg) & ~31, r0 = (8 * sg) & 31;
    const int pa = kq_off(c, col0 + perm32(r0)), pb = kq_off(c, col0 + perm32(r0 + 4));
    *reinterpret_cast<uint2*>(cb.K + pa) = uint2{f.k[it].x, f.k[it].y};
    *reinterpret_cast<uint2*>(cb.K + pb) = uint2{f.k[it].z, f.k[it].w};
    *reinterpret_cast<uint2*>(cb.Q + pa) = uint2{f.q[it].x, f.q[it].y};
    *reinterpret_cast<uint2*>(cb.Q + pb) = uint2{f.q[it].z, f.q[it].w};
  }
}

// Unit g of a chunk's gates (beta, e^gamma, e^{gamma_last - gamma}; 16 units each),
// as an offset from beta, so that the address stays a known LDS address.
__device__ __forceinline__ float* gate_unit(const ChunkBufs& cb, int g) {
  return cb.bet + (g >> 4) * (2 * C) + 4 * (g & 15);
}

// Persistent kernel: the number of chains in the workgroup's list, and the first
// chain at or after position k that has tokens (chain_count if none).
template <class Smem>
__device__ __forceinline__ int chain_count(Smem& sm) {
  return min(sm.pcount, kMaxPersistList);
}

template <class Smem>
__device__ __forceinline__ int next_chain(Smem& sm, int k) {
  const int n = chain_count(sm);
  while (k < n && sm.ps1[k] <= sm.ps0[k]) ++k;
  return k;
}

// The producer loop: chunk t is prepared into the buffers of parity t & 1 once the
// consumers are done with the chunk that used them last (chunk t - 2).  The four producer waves meet twice per chunk
// (after staging; after the tiles and diagonal blocks) on their own counter; the
// chunk is handed over when all four are done.  V is staged for the workgroup's
// state rows [row0, row0 + ROWS) only.
template <class V, class Smem>
__device__ __forceinline__ void producer_loop(Smem& sm, const PrefillArgs& p, int64_t s0, int64_t s1,
                                              int nchunks, int h, int hq, int hk, int row0, int pw, int lane0) {
  constexpr int NVIT = (V::VSEG + NPROD - 1) / NPROD;  // V segments per producer thread
  const int pt = pw * 64 + lane0;
  const float neg_decay = -expf(p.A_log[h]);
  const float dt_bias = p.dt_bias[h];
  const LaneOffsets lo = {(pt >> 4) * p.Hk * D + 8 * (pt & 15), (pt >> 4) * p.Hq * D + 8 * (pt & 15), pt * p.Hv};
  // V slice: segment pt + 256 it is token c, columns row0 + 8 sg .. +7.
  int voff[NVIT], vrow[NVIT];
#pragma unroll
  for (int it = 0; it < NVIT; ++it) {
    const int seg = pt + it * NPROD, c = seg / (V::ROWS / 8), sg = seg % (V::ROWS / 8);
    vrow[it] = seg < V::VSEG ? c : C;  // C: no segment
    voff[it] = c * p.Hv * D + 8 * sg;
  }
  static_assert(V::NP == 4 && !V::kPipelined, "pipelined producers run producer_loop_split");
  // The persistent kernel runs the chains of the workgroup's list (chain k covers
  // tokens [s0, s1)) as one stream of chunks; u counts the chunks of the stream and
  // indexes the hand-offs and the buffer parities (u = t otherwise).  Chain 0
  // (the longest of the list) is known before the rest of the list, which is
  // waited for (kList) where the stream first looks past a chain.
  int k = 0;
  bool listed = false;
  if constexpr (V::kPersist) {
    s0 = sm.ps0[0];
    s1 = sm.ps1[0];
    nchunks = int((s1 - s0 + C - 1) / C);
    if (nchunks == 0) return;  // the longest chain is empty: so are the others
  }
  ProducerPrefetch f;
  uint4 fv[NVIT];
  producer_prefetch(p, s0, int(s1 - s0 < C ? s1 - s0 : C), h, hq, hk, pt, lo, f);
  // The first wave forms each chunk's gates one tick ahead (chunk t + 1's in step 3
  // of tick t, where it has slack) and stores them with the chunk's K and Q.
  ChunkGates gts = {0.f, 0.f, 0.f, 0.f, 0.f};
  if (pw == 0) gts = chunk_gates(f, lane0, int(s1 - s0 < C ? s1 - s0 : C), neg_decay, dt_bias);

  int u = 0;
  for (;;) {
  for (int t = 0; t < nchunks; ++t, ++u) {
    // The lane index is re-materialised opaquely each tick so that lane-dependent
    // LDS addresses are recomputed in the loop rather than hoisted and spilled.
    int lane = lane0;
    asm volatile("" : "+v"(lane));
    const int64_t cs = s0 + int64_t(t) * C;
    const int clen = int(s1 - cs < C ? s1 - cs : C);
    // The next chunk: this chain's, or (persistent) the next chain's first.
    int64_t ncs = cs + C;
    int nclen = int(s1 - ncs < C ? s1 - ncs : C);
    bool has_next = ncs < s1;
    if constexpr (V::kPersist) {
      if (!has_next) {
        if (!listed) {
          wait_count<V::kHooks>(sm, kList, 1);
          listed = true;
        }
        const int nk = next_chain(sm, k + 1);
        if (nk < chain_count(sm)) {
          has_next = true;
          ncs = sm.ps0[nk];
          nclen = int(sm.ps1[nk] - ncs < C ? sm.ps1[nk] - ncs : C);
        }
      }
    }
    const ChunkBufs cb = chunk_bufs(sm, u & 1);
    // The buffers of chunk u - 2 (the same ones) consumed.
    if (u >= 2) wait_count<V::kHooks>(sm, kConsumed, V::NCW * (u - 1));

    // 1: stage K/Q (permuted columns), gates
    stage_kq(cb, f, pt);
    if (pw == 0) store_gates(cb, gts, lane);
    // The V slice of this chunk into registers; staged at the end of the tick,
    // after the consumers' last read of the previous chunk's V.
    {
      const uint16_t* vb = p.v + (cs * p.Hv + h) * D + row0;
#pragma unroll
      for (int it = 0; it < NVIT; ++it) {
        fv[it] = uint4{0u, 0u, 0u, 0u};
        if (vrow[it] < clen) fv[it] = *reinterpret_cast<const uint4*>(vb + voff[it]);
      }
    }
    signal_count(sm, kPPhase, lane);
    wait_count<V::kHooks>(sm, kPPhase, 4 * (2 * u + 1));  // all of K/Q/gates staged
    // The rest of the chunk is the longer chain: producer waves go ahead of the
    // consumer wave sharing the SIMD.
    __builtin_amdgcn_s_setprio(1);

    // 2: the next chunk's K/Q loads; diagonal N tiles (the solve waits for
    // them); then the diagonal blocks of T~ (wave 0) or the off-diagonal N tiles
    // and two P tiles each (the others, in the solve's shadow: P does not depend
    // on T~).
    // Split variants (few chains, a light consumer) put the solve first: the
    // other waves issue their loads after their diagonal tile, the solve wave
    // after its solve.
    constexpr bool kSolveFirst = V::F > 1;
    if (!kSolveFirst && has_next) producer_prefetch(p, ncs, nclen, h, hq, hk, pt, lo, f);
    switch (pw) {
      case 0:
        diag_tiles<0, 1>(sm, cb, lane);
        signal_count(sm, kDiagN, lane);
        wait_count<V::kHooks>(sm, kDiagN, 4 * (u + 1));
        diag_solve(sm, cb, lane);
        break;
      case 1: {
        diag_tiles<1, 2>(sm, cb, lane);
        signal_count(sm, kDiagN, lane);
        if (kSolveFirst && has_next) producer_prefetch(p, ncs, nclen, h, hq, hk, pt, lo, f);
        const TileJob j1[2] = {{1, 1, 0}, {1, 2, 0}};
        run_tiles(sm, cb, j1, p.scale, lane);
        const TileJob j2[2] = {{2, 0, 0}, {2, 3, 3}};
        run_tiles(sm, cb, j2, p.scale, lane);
        break;
      }
      case 2: {
        diag_tiles<2, 3>(sm, cb, lane);
        signal_count(sm, kDiagN, lane);
        if (kSolveFirst && has_next) producer_prefetch(p, ncs, nclen, h, hq, hk, pt, lo, f);
        const TileJob j1[2] = {{1, 3, 0}, {1, 2, 1}};
        run_tiles(sm, cb, j1, p.scale, lane);
        const TileJob j2[2] = {{2, 1, 0}, {2, 3, 0}};
        run_tiles(sm, cb, j2, p.scale, lane);
        break;
      }
      default: {
        diag_tiles<3, 4>(sm, cb, lane);
        signal_count(sm, kDiagN, lane);
        if (kSolveFirst && has_next) producer_prefetch(p, ncs, nclen, h, hq, hk, pt, lo, f);
        const TileJob j1[2] = {{1, 3, 1}, {1, 3, 2}};
        run_tiles(sm, cb, j1, p.scale, lane);
        const TileJob j2[2] = {{2, 1, 1}, {2, 2, 0}};
        run_tiles(sm, cb, j2, p.scale, lane);
        break;
      }
    }
    signal_count(sm, kPPhase, lane);
    wait_count<V::kHooks>(sm, kPPhase, 4 * (2 * u + 2));  // diagonal blocks and N tiles done

    // 3: off-diagonal blocks of T~ (waves 1 and 3), the remaining P tiles (two
    // each on waves 0 and 2), V once the consumers have read the previous chunk's
    switch (pw) {
      case 0: {
        if (kSolveFirst && has_next) producer_prefetch(p, ncs, nclen, h, hq, hk, pt, lo, f);
        const TileJob j1[2] = {{2, 2, 1}, {2, 2, 2}};
        run_tiles(sm, cb, j1, p.scale, lane);
        if (has_next) gts = chunk_gates(f, lane, nclen, neg_decay, dt_bias);  // the next chunk's gates
        break;
      }
      case 1: {
        offdiag_right(sm, cb, u, lane);
        break;
      }
      case 2: {
        const TileJob j1[2] = {{2, 3, 1}, {2, 3, 2}};
        run_tiles(sm, cb, j1, p.scale, lane);
        break;
      }
      default:
        offdiag_left<V::kHooks>(sm, cb, u, lane);
        break;
    }
    if (u >= 1) wait_count<V::kHooks>(sm, kVFree, V::NCW * u);
#pragma unroll
    for (int it = 0; it < NVIT; ++it) {
      const int seg = pt + it * NPROD;
      if (seg < V::VSEG)
        *reinterpret_cast<uint4*>(sm.V + (seg / (V::ROWS / 8)) * VSTR + 8 * (seg % (V::ROWS / 8))) = fv[it];
    }
    __builtin_amdgcn_s_setprio(0);
    if (!V::kHooks || p.ready_chunks <= 0 || t < p.ready_chunks) signal_count(sm, kReady, lane);
  }
  if constexpr (!V::kPersist) {
    break;
  } else {
    k = next_chain(sm, k + 1);
    if (k >= chain_count(sm)) break;
    s0 = sm.ps0[k];
    s1 = sm.ps1[k];
    nchunks = int((s1 - s0 + C - 1) / C);
  }
  }
}

// The raw gate inputs (a, b) of token `lane` of a chunk, clamped into the chunk.
template <int NT>
__device__ __forceinline__ void prefetch_gate_inputs(const PrefillArgs& p, int64_t cs, int clen, int h, int lane,
                                                     ProducerPrefetchT<NT>& f) {
  const int off = (lane < clen ? lane : clen - 1) * p.Hv;
  f.a = (p.a + cs * p.Hv + h)[off];
  f.b = (p.b + cs * p.Hv + h)[off];
}

template <int SI, class Smem>
__device__ __forceinline__ void diag_tile_of(Smem& sm, const ChunkBufs& cb, int lane) {
  diag_tiles<SI, SI + 1>(sm, cb, lane);
}

// The producer loop of split chains, pipelined one step deep: seven producer
// waves beside one consumer (chains split 8 ways) or six beside two (split 4
// ways), with NS = NP - 3 of them stagers.  For chunk t:
//   * wave 0 solves the diagonal blocks of T~ once chunk t's four diagonal N tiles
//     are in, then forms chunk t + 1's gates (and, with three stagers, chunk t + 1's
//     last diagonal N tile);
//   * waves 1 and 3 form the six off-diagonal N tiles (and one P tile each), then
//     the off-diagonal blocks of T~ (offdiag_right, offdiag_left);
//   * the stager waves (2, 4, 5[, 6]) form the other eight P tiles and stage V, then
//     stage chunk t + 1's K and Q and form its other diagonal N tiles,
// so the solve of chunk t + 1 can start as soon as chunk t's is done, instead of
// after chunk t + 1's staging and diagonal tiles.  Hand-offs per chunk: kStaged
// NS + 1 (the stagers' K/Q and wave 0's gates), kVStaged NS, kDiagN 4, kPPhase 3
// (the solve, and the N tiles of waves 1 and 3), kNRead 1 (the left off-diagonal
// wave read its N operands, so the next chunk's N tiles may overwrite them), kX32
// 1, kReady NS + 2 (waves 1 and 3, the stagers).  Every buffer of chunk t + 1's
// parity is written only after the consumers signalled chunk t - 1 consumed.
template <class V>
__device__ __forceinline__ void producer_loop_split(PrefillSmem& sm, const PrefillArgs& p, int64_t s0, int64_t s1,
                                                    int nchunks, int h, int hq, int hk, int row0, int pw,
                                                    int lane0) {
  static_assert(V::kPipelined && !V::kLoad, "pipelined producer loop of split chains");
  constexpr int NS = V::kStagers, NST = 64 * NS;        // stager waves, threads
  constexpr int NVIT = (V::VSEG + NST - 1) / NST;       // V segments per stager thread
  const int si = pw == 2 ? 0 : pw >= 4 ? pw - 3 : -1;   // stager index (waves 2, 4, 5, 6)
  const int pt = (si < 0 ? 0 : si) * 64 + lane0;        // thread index among the stagers
  const float neg_decay = -expf(p.A_log[h]);
  const float dt_bias = p.dt_bias[h];
  const LaneOffsets lo = {(pt >> 4) * p.Hk * D + 8 * (pt & 15), (pt >> 4) * p.Hq * D + 8 * (pt & 15), pt * p.Hv};
  int voff[NVIT], vrow[NVIT];
#pragma unroll
  for (int it = 0; it < NVIT; ++it) {
    const int seg = pt + it * NST, c = seg / (V::ROWS / 8), sg = seg % (V::ROWS / 8);
    vrow[it] = seg < V::VSEG ? c : C;  // C: no segment
    voff[it] = c * p.Hv * D + 8 * sg;
  }
  auto chunk_len = [&](int64_t cs) { return int(s1 - cs < C ? s1 - cs : C); };
  auto load_v = [&](uint4 (&fv)[NVIT], int64_t cs) {
    const uint16_t* vb = p.v + (cs * p.Hv + h) * D + row0;
    const int clen = chunk_len(cs);
#pragma unroll
    for (int it = 0; it < NVIT; ++it) {
      fv[it] = uint4{0u, 0u, 0u, 0u};
      if (vrow[it] < clen) fv[it] = *reinterpret_cast<const uint4*>(vb + voff[it]);
    }
  };
  // Diagonal N tiles: stager si forms tile si; with three stagers wave 0 forms tile 3.
  auto diag_tile = [&](const ChunkBufs& cb, int lane) {
    switch (si) {
      case 0: diag_tile_of<0>(sm, cb, lane); break;
      case 1: diag_tile_of<1>(sm, cb, lane); break;
      case 2: diag_tile_of<2>(sm, cb, lane); break;
      default: diag_tile_of<3>(sm, cb, lane); break;
    }
  };
  auto ready = [&](int t, int lane) {
    if (!V::kHooks || p.ready_chunks <= 0 || t < p.ready_chunks) signal_count(sm, kReady, lane);
  };
  // The stagers' eight P tiles (P(2,2) and P(3,3) go to waves 3 and 1).
  auto stager_tiles = [&](const ChunkBufs& cb, int lane) {
    if constexpr (NS == 4) {
      const TileJob jobs[4][2] = {{{2, 0, 0}, {2, 1, 0}}, {{2, 1, 1}, {2, 2, 0}}, {{2, 2, 1}, {2, 3, 0}},
                                  {{2, 3, 1}, {2, 3, 2}}};
      switch (si) {
        case 0: run_tiles(sm, cb, jobs[0], p.scale, lane); break;
        case 1: run_tiles(sm, cb, jobs[1], p.scale, lane); break;
        case 2: run_tiles(sm, cb, jobs[2], p.scale, lane); break;
        default: run_tiles(sm, cb, jobs[3], p.scale, lane); break;
      }
    } else {
      static_assert(NS == 3, "three or four stagers");
      const TileJob a0[2] = {{2, 0, 0}, {2, 1, 0}}, a1[1] = {{2, 1, 1}};
      const TileJob b0[2] = {{2, 2, 0}, {2, 2, 1}}, b1[1] = {{2, 3, 0}};
      const TileJob c0[2] = {{2, 3, 1}, {2, 3, 2}};
      switch (si) {
        case 0: run_tiles(sm, cb, a0, p.scale, lane); run_tiles(sm, cb, a1, p.scale, lane); break;
        case 1: run_tiles(sm, cb, b0, p.scale, lane); run_tiles(sm, cb, b1, p.scale, lane); break;
        default: run_tiles(sm, cb, c0, p.scale, lane); break;
      }
    }
  };

  ProducerPrefetchT<NST> f = {};
  uint4 fv[NVIT];
  // Chunk 0 ahead of the loop: its gates, K/Q, and diagonal N tiles.
  if (pw == 0) {
    prefetch_gate_inputs(p, s0, chunk_len(s0), h, lane0, f);
    store_gates(chunk_bufs(sm, 0), chunk_gates(f, lane0, chunk_len(s0), neg_decay, dt_bias), lane0);
    signal_count(sm, kStaged, lane0);
    if (nchunks > 1) prefetch_gate_inputs(p, s0 + C, chunk_len(s0 + C), h, lane0, f);
    if constexpr (NS == 3) {
      wait_count<V::kHooks>(sm, kStaged, NS + 1);
      diag_tile_of<3>(sm, chunk_bufs(sm, 0), lane0);
      signal_count(sm, kDiagN, lane0);
    }
  } else if (si >= 0) {
    producer_prefetch(p, s0, chunk_len(s0), h, hq, hk, pt, lo, f);
    load_v(fv, s0);
    stage_kq(chunk_bufs(sm, 0), f, pt);
    signal_count(sm, kStaged, lane0);
    if (nchunks > 1) producer_prefetch(p, s0 + C, chunk_len(s0 + C), h, hq, hk, pt, lo, f);
    wait_count<V::kHooks>(sm, kStaged, NS + 1);
    diag_tile(chunk_bufs(sm, 0), lane0);
    signal_count(sm, kDiagN, lane0);
  }

  for (int t = 0; t < nchunks; ++t) {
    int lane = lane0;
    asm volatile("" : "+v"(lane));
    const int64_t cs = s0 + int64_t(t) * C;
    const int64_t ncs = cs + C;
    const ChunkBufs cb = chunk_bufs(sm, t & 1);
    __builtin_amdgcn_s_setprio(1);
    switch (pw) {
      case 0:
        wait_count<V::kHooks>(sm, kDiagN, 4 * (t + 1));
        diag_solve(sm, cb, lane);
        signal_count(sm, kPPhase, lane);
        if (ncs < s1) {
          // Chunk t + 1's gates, stored into the buffers of chunk t - 1 once consumed.
          const ChunkGates g = chunk_gates(f, lane, chunk_len(ncs), neg_decay, dt_bias);
          if (t >= 1) wait_count<V::kHooks>(sm, kConsumed, V::NCW * t);
          const ChunkBufs cbn = chunk_bufs(sm, (t + 1) & 1);
          store_gates(cbn, g, lane);
          signal_count(sm, kStaged, lane);
          if (ncs + C < s1) prefetch_gate_inputs(p, ncs + C, chunk_len(ncs + C), h, lane, f);
          if constexpr (NS == 3) {
            // Chunk t + 1's last diagonal N tile, once its K is staged (the solve of
            // chunk t, just done, freed the scratch).
            wait_count<V::kHooks>(sm, kStaged, (NS + 1) * (t + 2));
            diag_tile_of<3>(sm, cbn, lane);
            signal_count(sm, kDiagN, lane);
          }
        }
        break;
      case 1: {
        wait_count<V::kHooks>(sm, kStaged, (NS + 1) * (t + 1));
        if (t >= 1) wait_count<V::kHooks>(sm, kNRead, t);  // chunk t - 1's N read by the left wave
        const TileJob j1[2] = {{1, 2, 1}, {1, 3, 2}};
        run_tiles(sm, cb, j1, p.scale, lane);
        const TileJob j2[2] = {{1, 3, 1}, {2, 3, 3}};
        run_tiles(sm, cb, j2, p.scale, lane);
        signal_count(sm, kPPhase, lane);
        wait_count<V::kHooks>(sm, kPPhase, 3 * (t + 1));
        offdiag_right(sm, cb, t, lane);
        ready(t, lane);
        break;
      }
      case 3: {
        wait_count<V::kHooks>(sm, kStaged, (NS + 1) * (t + 1));
        const TileJob j1[2] = {{1, 1, 0}, {1, 2, 0}};
        run_tiles(sm, cb, j1, p.scale, lane);
        const TileJob j2[2] = {{1, 3, 0}, {2, 2, 2}};
        run_tiles(sm, cb, j2, p.scale, lane);
        signal_count(sm, kPPhase, lane);
        wait_count<V::kHooks>(sm, kPPhase, 3 * (t + 1));
        offdiag_left<V::kHooks, true>(sm, cb, t, lane);
        ready(t, lane);
        break;
      }
      default: {  // stagers
        // Chunk t's V as soon as the consumers have read chunk t - 1's: with K, Q and
        // the gates (staged a tick ahead) it is all their retrieve and Y need.
        if (t >= 1) wait_count<V::kHooks>(sm, kVFree, V::NCW * t);
#pragma unroll
        for (int it = 0; it < NVIT; ++it) {
          const int seg = pt + it * NST;
          if (seg < V::VSEG)
            *reinterpret_cast<uint4*>(sm.V + (seg / (V::ROWS / 8)) * VSTR + 8 * (seg % (V::ROWS / 8))) = fv[it];
        }
        signal_count(sm, kVStaged, lane);
        if (ncs < s1) load_v(fv, ncs);  // chunk t + 1's V into registers
        wait_count<V::kHooks>(sm, kStaged, (NS + 1) * (t + 1));  // chunk t's gates (wave 0)
        stager_tiles(cb, lane);
        ready(t, lane);  // chunk t's P tiles
        if (ncs < s1) {
          // Chunk t + 1: K and Q into the buffers of chunk t - 1 once consumed; its
          // diagonal N tiles once the solve of chunk t freed their scratch.
          if (t >= 1) wait_count<V::kHooks>(sm, kConsumed, V::NCW * t);
          const ChunkBufs cbn = chunk_bufs(sm, (t + 1) & 1);
          stage_kq(cbn, f, pt);
          signal_count(sm, kStaged, lane);
          if (ncs + C < s1) producer_prefetch(p, ncs + C, chunk_len(ncs + C), h, hq, hk, pt, lo, f);
          wait_count<V::kHooks>(sm, kStaged, (NS + 1) * (t + 2));
          wait_count<V::kHooks>(sm, kPPhase, 3 * (t + 1));
          diag_tile(cbn, lane);
          signal_count(sm, kDiagN, lane);
        }
        break;
      }
    }
    __builtin_amdgcn_s_setprio(0);
  }
}

// The loader loop of the two-kernel path: the producers' hand-offs and staging,
// with chunk t's T~ (hi, lo), P and gates copied from their prepared images (tiles
// = image of chunk 0 of this chain; chunk t is Hv images further) instead of
// computed.  K and Q are staged as the producers stage them, V at the end of the
// tick, after the consumers' last read of the previous chunk's V.
// The images of chunk t + 1 are loaded into registers during tick t, so their
// latency overlaps the waits for the consumers.
// V goes two chunks ahead in every variant (two register sets): the prep kernel does
// not read V, so with inputs that the caches do not hold its loads come from HBM
// (one 4,096-token sequence, four rotating input sets: 142.5 -> 132.0 us, unchanged with one).
template <class V>
__device__ __forceinline__ void loader_loop(PrefillSmem& sm, const PrefillArgs& p, const u32x4* tiles, int64_t s0,
                                            int64_t s1, int nchunks, int h, int hq, int hk, int row0, int pw,
                                            int lane0) {
  constexpr int NVIT = (V::VSEG + NPROD - 1) / NPROD;        // V segments per loader thread
  constexpr int NTIT = (kTileImage + NPROD - 1) / NPROD;     // 16-byte tile units per loader thread
  constexpr int NT1 = kTileUnits1;                           // 16-byte units per tile image
  const int pt = pw * 64 + lane0;
  const LaneOffsets lo = {(pt >> 4) * p.Hk * D + 8 * (pt & 15), (pt >> 4) * p.Hq * D + 8 * (pt & 15), pt * p.Hv};
  int voff[NVIT], vrow[NVIT];
#pragma unroll
  for (int it = 0; it < NVIT; ++it) {
    const int seg = pt + it * NPROD, c = seg / (V::ROWS / 8), sg = seg % (V::ROWS / 8);
    vrow[it] = seg < V::VSEG ? c : C;  // C: no segment
    voff[it] = c * p.Hv * D + 8 * sg;
  }
  // Unit pt + 256 it of a chunk's images (the last round's excess lanes re-read
  // the last unit and store nothing).
  int toff[NTIT];
#pragma unroll
  for (int it = 0; it < NTIT; ++it) toff[it] = pt + it * NPROD < kTileImage ? pt + it * NPROD : kTileImage - 1;
  // (First-class vectors: copies of uint4 structs would go through the stack.)
  u32x4 tv[NTIT], fva[NVIT], fvb[NVIT];
  // V slice of chunk t (tokens [s0 + C t, s1) of it) into fv, zero past the sequence.
  auto load_v = [&](int t, u32x4(&fv)[NVIT]) {
    const int64_t vs = s0 + int64_t(t) * C;
    const int vlen = int(s1 - vs < C ? s1 - vs : C);
    const uint16_t* vb = p.v + (vs * p.Hv + h) * D + row0;
#pragma unroll
    for (int it = 0; it < NVIT; ++it) {
      fv[it] = u32x4{0u, 0u, 0u, 0u};
      if (vrow[it] < vlen) fv[it] = *reinterpret_cast<const u32x4*>(vb + voff[it]);
    }
  };
  ProducerPrefetch f;
  producer_prefetch(p, s0, int(s1 - s0 < C ? s1 - s0 : C), h, hq, hk, pt, lo, f);
  // Chunk 0's images, and the V slices of chunks 0 and 1, into registers.
#pragma unroll
  for (int it = 0; it < NTIT; ++it) tv[it] = tiles[toff[it]];
  load_v(0, fva);
  if (nchunks > 1) load_v(1, fvb);

  // Tick t stages chunk t from the registers tv (images) and fv (V), then loads
  // chunk t + 2's V into fv (the V loads go two chunks ahead, so that their latency
  // from HBM, when the inputs are not in the caches, stays off the chain).
  auto tick = [&](int t, u32x4(&fv)[NVIT]) {
    int lane = lane0;
    asm volatile("" : "+v"(lane));
    const int64_t cs = s0 + int64_t(t) * C;
    const int64_t ncs = cs + C;
    const int nclen = int(s1 - ncs < C ? s1 - ncs : C);
    const ChunkBufs cb = chunk_bufs(sm, t & 1);
    if (t >= 2) wait_count<V::kHooks>(sm, kConsumed, V::NCW * (t - 1));  // chunk t - 2 consumed
    stage_kq(cb, f, pt);
#pragma unroll
    for (int it = 0; it < NTIT; ++it) {
      const int e = pt + it * NPROD;
      if (e < kTileUnits) {
        uint16_t* dst = e < NT1       ? cb.Th + 8 * e
                        : e < 2 * NT1 ? cb.Tl + 8 * (e - NT1)
                                      : cb.P + 8 * (e - 2 * NT1);
        *reinterpret_cast<u32x4*>(dst) = tv[it];
      } else if (e < kTileImage) {
        *reinterpret_cast<u32x4*>(gate_unit(cb, e - kTileUnits)) = tv[it];
      }
    }
    if (t >= 1) wait_count<V::kHooks>(sm, kVFree, V::NCW * t);  // the consumers' last read of V
#pragma unroll
    for (int it = 0; it < NVIT; ++it) {
      const int seg = pt + it * NPROD;
      if (seg < V::VSEG)
        *reinterpret_cast<u32x4*>(sm.V + (seg / (V::ROWS / 8)) * VSTR + 8 * (seg % (V::ROWS / 8))) = fv[it];
    }
    if (!V::kHooks || p.ready_chunks <= 0 || t < p.ready_chunks) signal_count(sm, kReady, lane);
    // The next chunks' loads go out after the hand-off.  Issued before it, the
    // waits for this tick's registers (loaded a tick earlier) would also wait for
    // them: the K/Q loads are conditional, so the compiler cannot count them and
    // waits for every load issued since.
    if (ncs < s1) producer_prefetch(p, ncs, nclen, h, hq, hk, pt, lo, f);
    if (t + 1 < nchunks) {  // chunk t + 1's images into registers
      const u32x4* src = tiles + int64_t(t + 1) * p.Hv * kTileImage;
#pragma unroll
      for (int it = 0; it < NTIT; ++it) tv[it] = src[toff[it]];
    }
    if (t + 2 < nchunks) load_v(t + 2, fv);  // chunk t + 2's V slice
  };
  for (int t = 0; t < nchunks; t += 2) {
    tick(t, fva);
    if (t + 1 < nchunks) tick(t + 1, fvb);
  }
}

// ---------------------------------------------------------------------------
// Consumer side (waves 0 .. NCW-1; wave w owns state rows R0 + VW w .. + VW - 1)
// ---------------------------------------------------------------------------

// Xk = K S^T (rows c, cols v) with S as hi/lo B operands, and Xq = (Q S^T)^T
// (rows v, cols c) with S's hi part as the A operand (output-only product).
template <int VT>
__device__ __forceinline__ void retrieve(const ChunkBufs& cb, const f32x4 (&S)[VT][8], f32x4 (&Xk)[4][VT],
                                         f32x4 (&Xq)[VT][4], int lane) {
#pragma unroll
  for (int ct = 0; ct < 4; ++ct)
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) Xk[ct][vt] = Xq[vt][ct] = zero4();
  if constexpr (VT == 1) {
    // One state tile leaves registers for the next contraction block's K and Q
    // fragments: they are read while this block's MFMAs run (the scheduling
    // barrier keeps the reads ahead of them).
    uint4 kf[2][4], qf[2][4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      kf[0][ct] = frag_kq(cb.K, 16 * ct, 0, lane);
      qf[0][ct] = frag_kq(cb.Q, 16 * ct, 0, lane);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) {
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
          kf[(ks + 1) & 1][ct] = frag_kq(cb.K, 16 * ct, ks + 1, lane);
          qf[(ks + 1) & 1][ct] = frag_kq(cb.Q, 16 * ct, ks + 1, lane);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      uint4 Sh, Sl;
      split_pack(S[0][2 * ks], S[0][2 * ks + 1], Sh, Sl);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        Xk[ct][0] = mfma(kf[ks & 1][ct], Sh, Xk[ct][0]);
        Xk[ct][0] = mfma(kf[ks & 1][ct], Sl, Xk[ct][0]);
        Xq[0][ct] = mfma(Sh, qf[ks & 1][ct], Xq[0][ct]);
      }
    }
    return;
  }
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    uint4 Sh[VT], Sl[VT];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) split_pack(S[vt][2 * ks], S[vt][2 * ks + 1], Sh[vt], Sl[vt]);
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const uint4 ak = frag_kq(cb.K, 16 * ct, ks, lane);
      const uint4 bq = frag_kq(cb.Q, 16 * ct, ks, lane);
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        Xk[ct][vt] = mfma(ak, Sh[vt], Xk[ct][vt]);
        Xk[ct][vt] = mfma(ak, Sl[vt], Xk[ct][vt]);
        Xq[vt][ct] = mfma(Sh[vt], bq, Xq[vt][ct]);
      }
    }
  }
}

// State row (within the wave's VW rows) held by column n of state tile vt.  With two
// tiles the rows interleave in groups of four (tile 0: 0-3, 8-11, ..., tile 1: 4-7,
// 12-15, ...), so that a lane's output rows of the two tiles are 8 consecutive values.
template <int VT>
__device__ __forceinline__ int vrow(int vt, int n) {
  return VT == 2 ? 8 * (n >> 2) + 4 * vt + (n & 3) : 16 * vt + n;
}

// The consumer loop: iteration t (>= 1) advances the state through chunk t-1
// from the buffers of parity (t-1) & 1, once the producers have handed it over.
// Column n of state tile vt is state row row0 + VW wave + vrow(vt, n) (V column
// VW wave + vrow(vt, n) of the staged slice).
template <class V>
__device__ __forceinline__ void consumer_loop(PrefillSmem& sm, const PrefillArgs& p, int64_t s0, int64_t s1,
                                              int nchunks, int h, int row0, int wave, int lane0,
                                              f32x4 (&S)[V::VT][8], int u0 = 0) {
  constexpr int VT = V::VT, VW = V::VW;
  const int64_t vstride = int64_t(p.Hv) * D;
  // Element offset of output row 16ct + lane%16, first column of the lane's output
  // values (8 (lane/16) with two state tiles, 4 (lane/16) with one), from the wave's
  // (uniform) chunk base.
  int orow[4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) orow[ct] = (16 * ct + (lane0 & 15)) * int(vstride) + (VT == 2 ? 8 : 4) * (lane0 >> 4);
  for (int t = 1; t <= nchunks; ++t) {
    int lane = lane0;
    asm volatile("" : "+v"(lane));
    const int g = lane >> 4, n16 = lane & 15;
    const int64_t cs = s0 + int64_t(t - 1) * C;
    const int clen = int(s1 - cs < C ? s1 - cs : C);
    // u: the chunk's position in the workgroup's stream of chunks (persistent
    // kernel: u0 chunks of earlier chains precede this chain's).
    const int u = u0 + t;
    const ChunkBufs cb = chunk_bufs(sm, (u - 1) & 1);
    if constexpr (V::kPipelined) {
      // Pipelined producers hand a chunk over in two steps: K, Q, the gates and V for
      // the retrieve and Y, then T~ and P ("ready", below) for v_new and the output.
      wait_count<V::kHooks>(sm, kStaged, (V::kStagers + 1) * u);
      wait_count<V::kHooks>(sm, kVStaged, V::kStagers * u);
    } else {
      wait_count<V::kHooks>(sm, kReady, 4 * u);  // chunk u - 1 prepared
    }

    // 1: X = K S^T, (Q S^T)^T
    f32x4 Xk[4][VT], Xq[VT][4];
    retrieve(cb, S, Xk, Xq, lane);

    // 2: Y, v_new, output
    // Y = beta (V - e^gamma X); element (c = 16ct + 4g + i, v = VW w + vrow(vt, n16)).
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const float4 bc = *reinterpret_cast<const float4*>(cb.bet + 16 * ct + 4 * g);
      const float4 ec = *reinterpret_cast<const float4*>(cb.eg + 16 * ct + 4 * g);
      const float b4[4] = {bc.x, bc.y, bc.z, bc.w}, e4[4] = {ec.x, ec.y, ec.z, ec.w};
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        // V rows 16ct + 4g .. +3 of column VW w + vrow(vt, n16): lane j of a 16-lane
        // group reads the 4 columns VW w + vrow(vt, 4 (j & 3)) .. +3 of row 16ct + 4g + j/4.
        const uint2 vv = read_tr(sm.V + (16 * ct + 4 * g + (n16 >> 2)) * VSTR + VW * wave + vrow<VT>(vt, 4 * (n16 & 3)));
        const float vf[4] = {bf16lo_f32(vv.x), bf16hi_f32(vv.x), bf16lo_f32(vv.y), bf16hi_f32(vv.y)};
#pragma unroll
        for (int i = 0; i < 4; ++i) Xk[ct][vt][i] = b4[i] * (vf[i] - e4[i] * Xk[ct][vt][i]);
      }
      const float ecn = cb.eg[16 * ct + n16] * p.scale;  // scale e^gamma of output column c = 16ct + n16
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) Xq[vt][ct] = Xq[vt][ct] * ecn;
    }
    signal_count(sm, kVFree, lane);  // V of this chunk read
    if constexpr (V::kPipelined) wait_count<V::kHooks>(sm, kReady, (V::kStagers + 2) * u);  // T~ and P
    // The 16-row consumer reads all its T~ and P operands now (they are ready), so that
    // their latency overlaps the Y split; the 32-row one, short of registers, as used.
    // Pair (ct, js) of T~ is fragment ct < 2 ? ct : 2 ct - 2 + js; pair (js, ct) of
    // P is fragment js ? ct + 2 : ct.
    constexpr int NPF = VT == 1 ? 6 : 1;
    uint4 thf[NPF], tlf[NPF], pqf[NPF];
    if constexpr (VT == 1) {
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int js = 0; js <= (ct >> 1); ++js) {
          const int i = ct < 2 ? ct : 2 * ct - 2 + js;
          thf[i] = tile_row<V::kLoad>(cb.Th, ct, js, lane);
          tlf[i] = tile_row<V::kLoad>(cb.Tl, ct, js, lane);
        }
#pragma unroll
      for (int js = 0; js < 2; ++js)
#pragma unroll
        for (int ct = 2 * js; ct < 4; ++ct) pqf[js ? ct + 2 : ct] = tile_row<V::kLoad>(cb.P, ct, js, lane);
      __builtin_amdgcn_sched_barrier(0);
    }
    // v_new = T~ Y (contraction over the rows of Y in blocks js; T~ is lower triangular).
    uint4 Yh[VT][2], Yl[VT][2];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int js = 0; js < 2; ++js) split_pack(Xk[2 * js][vt], Xk[2 * js + 1][vt], Yh[vt][js], Yl[vt][js]);
    f32x4 Vn[4][VT];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) Vn[ct][vt] = zero4();
#pragma unroll
      for (int js = 0; js <= (ct >> 1); ++js) {
        uint4 th, tl;
        if constexpr (VT == 1) {
          th = thf[ct < 2 ? ct : 2 * ct - 2 + js];
          tl = tlf[ct < 2 ? ct : 2 * ct - 2 + js];
        } else {
          th = tile_row<V::kLoad>(cb.Th, ct, js, lane);
          tl = tile_row<V::kLoad>(cb.Tl, ct, js, lane);
        }
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          Vn[ct][vt] = mfma(th, Yh[vt][js], Vn[ct][vt]);
          Vn[ct][vt] = mfma(th, Yl[vt][js], Vn[ct][vt]);
          Vn[ct][vt] = mfma(tl, Yh[vt][js], Vn[ct][vt]);
        }
      }
    }
    // o^T = scale e^gamma (S Q^T) + v_new^T (scale P)^T (rows v, cols c); P is lower triangular.
#pragma unroll
    for (int js = 0; js < 2; ++js) {
      uint4 vb[VT];
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) vb[vt] = pack_hi(Vn[2 * js][vt], Vn[2 * js + 1][vt]);
#pragma unroll
      for (int ct = 2 * js; ct < 4; ++ct) {
        uint4 pq;
        if constexpr (VT == 1) {
          pq = pqf[js ? ct + 2 : ct];
        } else {
          pq = tile_row<V::kLoad>(cb.P, ct, js, lane);
        }
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) Xq[vt][ct] = mfma(vb[vt], pq, Xq[vt][ct]);
      }
    }
    // 3: S = e^{gamma_last} S + sum_c K[c]^T (d_c v_new[c]),  d_c = e^{gamma_last - gamma_c}
    const float dlast = cb.eg[clen - 1];
    uint4 Uh[VT][2], Ul[VT][2];
#pragma unroll
    for (int js = 0; js < 2; ++js) {
      const float4 d0 = *reinterpret_cast<const float4*>(cb.dd + 32 * js + 4 * g);
      const float4 d1 = *reinterpret_cast<const float4*>(cb.dd + 32 * js + 16 + 4 * g);
      const f32x4 e0 = {d0.x, d0.y, d0.z, d0.w}, e1 = {d1.x, d1.y, d1.z, d1.w};
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) split_pack(Vn[2 * js][vt] * e0, Vn[2 * js + 1][vt] * e1, Uh[vt][js], Ul[vt][js]);
    }
    const KtBases kb = kt_bases(lane);
    static_for<8>([&](auto KT) {
      constexpr int kt = decltype(KT)::value;
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) S[vt][kt] = S[vt][kt] * dlast;
      static_for<2>([&](auto JS) {
        constexpr int js = decltype(JS)::value;
        const uint4 ak = frag_tr_k_at<js, kt>(cb.K, kb);
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          S[vt][kt] = mfma(ak, Uh[vt][js], S[vt][kt]);
          S[vt][kt] = mfma(ak, Ul[vt][js], S[vt][kt]);
        }
      });
    });
    // The output stores, in the same block as the state update so that their packing
    // and issue fill the update's MFMA shadow.  Lane holds o[c = 16ct + n16][v = row0 +
    // VW w + vrow(vt, 4g + i)]: with two tiles 8 consecutive v (one 16-byte store per
    // ct), with one 4 (8 bytes).  Rows at or past clen fall outside the buffer
    // resource, whose extent ends at the chunk's last token: the hardware drops their
    // stores, so no lane needs a branch.
    {
      const BufferRsrc orsrc = buffer_rsrc(p.out + cs * vstride + (int64_t(h) * D + row0 + VW * wave),
                                           uint32_t(clen) * uint32_t(vstride) * 2u);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        if constexpr (VT == 2) {
          const f32x4 &o0 = Xq[0][ct], &o1 = Xq[1][ct];
          buffer_store16(u32x4{pack_bf16x2(o0[0], o0[1]), pack_bf16x2(o0[2], o0[3]), pack_bf16x2(o1[0], o1[1]),
                               pack_bf16x2(o1[2], o1[3])},
                         orsrc, 2 * orow[ct]);
        } else {
          const f32x4& o = Xq[0][ct];
          buffer_store8(u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])}, orsrc, 2 * orow[ct]);
        }
      }
    }
    signal_count(sm, kConsumed, lane);  // buffers of this chunk no longer read
  }
}

// The sequence of rank `rank` in descending length order (ties: lower index
// first), so the longest chains start first; natural order for large batches.  `len` and
// `picked` are LDS scratch (up to kMaxSortedSeqs lengths, and the result).
template <int NTHREADS>
__device__ int pick_sequence(int* len, int* picked, const PrefillArgs& p, int rank, int tid) {
  if (p.N <= 1 || p.N > kMaxSortedSeqs) return rank;
  for (int i = tid; i < p.N; i += NTHREADS) {
    int64_t a = load_cu(p.cu_seqlens, p.cu_is_64, i), b = load_cu(p.cu_seqlens, p.cu_is_64, i + 1);
    a = a < 0 ? 0 : (a > p.T ? p.T : a);
    b = b < a ? a : (b > p.T ? p.T : b);
    len[i] = int(b - a);
  }
  __syncthreads();
  for (int i = tid; i < p.N; i += NTHREADS) {
    const int li = len[i];
    int r = 0;
    for (int j = 0; j < p.N; ++j) {
      const int lj = len[j];
      r += (lj > li) | ((lj == li) & (j < i));
    }
    if (r == rank) *picked = i;
  }
  __syncthreads();
  return *picked;
}

// Workgroup b handles slice f of chain `chain` (chain = rank-major, v-head
// minor).  With F > 1 the F slices of chain c are b = 16 F (c / 16) + 8 (F (c % 2)
// + f) + (c % 16) / 2: workgroups are dealt to the XCDs round-robin, so the slices
// of one chain, and those of its GQA partner (chain c ^ 1), share an XCD (and its
// L2) for their common K/Q reads.  With F == 1 the two chains of a GQA pair share an
// XCD the same way.
template <class V>
__global__ __launch_bounds__(V::NTHREADS) void gdn_prefill_kernel(PrefillArgs p) {
  constexpr int NCW = V::NCW, VT = V::VT, VW = V::VW, NTHREADS = V::NTHREADS;
  __shared__ PrefillSmem sm;

  const int tid = threadIdx.x;
  const int lane0 = tid & 63;
  const int hw = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Role index.  Waves are dealt to the four SIMDs round-robin.  With four producers or
  // loaders the natural order measured as fast or faster (two consumers on SIMDs of their
  // own: +1.5%; the producer variant's solve wave sharing a SIMD: +7%).
  // With seven producers (beside one consumer) the consumer keeps hardware wave 0 and
  // shares its SIMD with the producer that has least to do (wave 0, the solve): hardware
  // waves 1-7 take producers 1, 2, 3, 0, 4, 5, 6.  With six (beside two consumers on
  // hardware waves 0 and 1) hardware waves 2-7 take producers 2, 3, 0, 5, 1, 4: the
  // consumers share their SIMDs with the solve wave and the third stager, and each
  // off-diagonal wave shares one with a stager (1.5-2.5% faster than pairing the
  // second consumer with the right off-diagonal wave, or the two off-diagonal waves).
  const int wave = V::NP == 7   ? (hw == 0 ? 0 : 1 + ((0x6540321 >> (4 * (hw - 1))) & 15))
                   : V::NP == 6 ? (hw < 2 ? hw : 2 + ((0x415032 >> (4 * (hw - 2))) & 15))
                                : hw;

  const int bid = blockIdx.x;
  // Workgroups are dealt to the 8 XCDs round-robin.  F == 1: blocks b and b + 8 of
  // each group of 16 take chains 2m and 2m + 1 (v-heads 2j, 2j + 1, which read the
  // same K and Q), so the two start together on one XCD and share its L2.  F > 1:
  // in each group of 16 F blocks, the 2 F blocks b = 8 l + x (l = 0 .. 2F - 1) of
  // XCD x take slice l % F of chain 2x + l / F: both chains of a pair, all slices.
  const int chain = V::F == 1 ? (bid & ~15) | ((bid & 7) << 1) | ((bid >> 3) & 1)
                              : (bid / (16 * V::F)) * 16 + 2 * (bid % 8) + (bid / 8) % (2 * V::F) / V::F;
  const int row0 = V::F == 1 ? 0 : ((bid / 8) % V::F) * V::ROWS;
  if (chain >= p.N * p.Hv) return;  // padding of the last group of 16 chains (workgroup-uniform)
  const int h = chain % p.Hv;
  const int seq = pick_sequence<NTHREADS>(reinterpret_cast<int*>(sm.Nh), &sm.seq, p, chain / p.Hv, tid);
  const int hq = h / (p.Hv / p.Hq);
  const int hk = h / (p.Hv / p.Hk);

  int64_t s0, s1;
  if constexpr (V::kLoad) {
    const SeqRange r = seq_range(p, seq);
    s0 = r.s0;
    s1 = r.s1;
  } else {
    s0 = load_cu(p.cu_seqlens, p.cu_is_64, seq);
    s1 = load_cu(p.cu_seqlens, p.cu_is_64, seq + 1);
    s0 = s0 < 0 ? 0 : (s0 > p.T ? p.T : s0);
    s1 = s1 < s0 ? s0 : (s1 > p.T ? p.T : s1);
  }
  const int nchunks = int((s1 - s0 + C - 1) / C);

  if (nchunks > 0) {
    // Blocks of T~, N and P that are never written per chunk are read as zeros
    // (strictly-upper blocks, the diagonal blocks of Nh/Nl): clear them once.
    // pick_sequence's last read of its scratch precedes its final barrier.
    const uint4 z = uint4{0u, 0u, 0u, 0u};
    for (int e = tid; e < C * TSTR / 8; e += NTHREADS) {
      reinterpret_cast<uint4*>(sm.P[0])[e] = z;
      reinterpret_cast<uint4*>(sm.P[1])[e] = z;
      reinterpret_cast<uint4*>(sm.Th[0])[e] = z;
      reinterpret_cast<uint4*>(sm.Th[1])[e] = z;
      reinterpret_cast<uint4*>(sm.Tl[0])[e] = z;
      reinterpret_cast<uint4*>(sm.Tl[1])[e] = z;
      if (e < NROWS * TSTR / 8) {
        reinterpret_cast<uint4*>(sm.Nh)[e] = z;
        reinterpret_cast<uint4*>(sm.Nl)[e] = z;
      }
    }
    if (tid < 16) sm.sync[tid] = 0;
    if (V::kHooks && tid == 0) {
      sm.spin_limit = p.spin_limit > 0 ? p.spin_limit : kSpinLimit;
      sm.aborts = p.aborts;
    }
  }
  __syncthreads();  // cleared LDS and counters visible to both roles

  if (wave >= NCW) {
    if (nchunks > 0) {
      if constexpr (V::kLoad) {
        const u32x4* tiles = reinterpret_cast<const u32x4*>(p.tiles) +
                             (int64_t(chunks_before(p, seq, lane0)) * p.Hv + h) * kTileImage;
        loader_loop<V>(sm, p, tiles, s0, s1, nchunks, h, hq, hk, row0, wave - NCW, lane0);
      } else {
        if constexpr (V::kPipelined) {
          producer_loop_split<V>(sm, p, s0, s1, nchunks, h, hq, hk, row0, wave - NCW, lane0);
        } else {
          producer_loop<V>(sm, p, s0, s1, nchunks, h, hq, hk, row0, wave - NCW, lane0);
        }
      }
    }
    return;
  }

  const int64_t state_head = (int64_t(seq) * p.Hv + h) * D * D;
  const int g = lane0 >> 4, n16 = lane0 & 15;
  // Consumer state slab: rows v = row0 + VW*wave + vrow(vt, n16), cols k = 16*kt + 4g + i.
  f32x4 S[VT][8];
#pragma unroll
  for (int vt = 0; vt < VT; ++vt) {
    const int v = row0 + VW * wave + vrow<VT>(vt, n16);
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
      if (p.state) {
        const float4 x = *reinterpret_cast<const float4*>(p.state + state_head + int64_t(v) * D + 16 * kt + 4 * g);
        S[vt][kt] = f32x4{x.x, x.y, x.z, x.w};
      } else {
        S[vt][kt] = zero4();
      }
    }
  }
  if (nchunks > 0) {
    consumer_loop<V>(sm, p, s0, s1, nchunks, h, row0, wave, lane0, S);
    if (aborted(sm)) {
      // A hand-off wait gave up: NaN over every output element of this wave (all
      // chunks of the sequence, its state rows of head h) and its state slice.
      const int64_t vstride = int64_t(p.Hv) * D;
      uint16_t* obase = p.out + int64_t(h) * D + row0 + VW * wave + (VT == 2 ? 8 : 4) * (lane0 >> 4);
      for (int64_t tok = s0 + n16; tok < s1; tok += 16) {
        if constexpr (VT == 2) {
          *reinterpret_cast<uint4*>(obase + tok * vstride) = uint4{kNaNx2, kNaNx2, kNaNx2, kNaNx2};
        } else {
          *reinterpret_cast<uint2*>(obase + tok * vstride) = uint2{kNaNx2, kNaNx2};
        }
      }
      const float nan = __builtin_nanf("");
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) S[vt][kt] = f32x4{nan, nan, nan, nan};
    }
  }

  // Final state (for an empty sequence: the initial state, or zeros).
  if (nchunks > 0 || p.state != p.new_state) {
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      const int v = row0 + VW * wave + vrow<VT>(vt, n16);
#pragma unroll
      for (int kt = 0; kt < 8; ++kt) {
        const f32x4 x = S[vt][kt];
        *reinterpret_cast<float4*>(p.new_state + state_head + int64_t(v) * D + 16 * kt + 4 * g) =
            make_float4(x[0], x[1], x[2], x[3]);
      }
    }
  }
}

// Minimum over the wave (uniform): DPP within each row of 16 lanes, then the four
// row minima.
__device__ __forceinline__ uint32_t wave_min(uint32_t x) {
  x = min(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0xB1, 0xF, 0xF, false)));
  x = min(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x4E, 0xF, 0xF, false)));
  x = min(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x124, 0xF, 0xF, false)));
  x = min(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x128, 0xF, 0xF, false)));
  const uint32_t a = uint32_t(__builtin_amdgcn_readlane(int(x), 0)), b = uint32_t(__builtin_amdgcn_readlane(int(x), 16));
  const uint32_t c = uint32_t(__builtin_amdgcn_readlane(int(x), 32)), d = uint32_t(__builtin_amdgcn_readlane(int(x), 48));
  return min(min(a, b), min(c, d));
}

// Persistent form of the F = 1 kernel, for batches of more chains than CUs: one
// workgroup per CU runs a list of whole chains back to back, so that the next
// chain's first chunk is loaded and prepared while the consumers finish the current
// one (a workgroup per chain pays for that, its start-up and its drain once per
// chain: about three chunk times).  The grid is B = gridDim.x / Hv bins of Hv
// workgroups; workgroup (bin, i) runs v-head h(i) of every sequence of its bin.
// Every workgroup forms the same schedule of the sequences over the bins, so all
// heads of a sequence share one bin and a bin's workgroups share their list: with
// LPT (at most kMaxPersistLpt sequences) longest-processing-time (longest first,
// each onto the least-loaded bin; cost 3 per chunk + 2 per sequence, ties to the
// lower bin), otherwise boustrophedon rounds over the longest-first order.
template <class V, bool LPT>
__global__ __launch_bounds__(V::NTHREADS) void gdn_prefill_persistent_kernel(PrefillArgs p) {
  static_assert(V::kPersist && V::NCW == 4 && V::VT == 2, "persistent kernel: Variant<4, 2, ..., true>");
  constexpr int NCW = V::NCW, VT = V::VT, VW = V::VW, NTHREADS = V::NTHREADS;
  __shared__ PrefillSmem sm;

  const int tid = threadIdx.x;
  const int lane0 = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bid = blockIdx.x;
  const int nbins = int(gridDim.x) / p.Hv, bin = bid / p.Hv, i = bid % p.Hv;
  // Workgroups are dealt to the 8 XCDs round-robin: with Hv a multiple of 16,
  // workgroups i and i + 8 of a bin (one XCD) take the GQA pair 2j, 2j + 1.
  const int h = p.Hv % 16 == 0 ? (i & ~15) | ((i & 7) << 1) | ((i >> 3) & 1) : i;
  const int hq = h / (p.Hv / p.Hq);
  const int hk = h / (p.Hv / p.Hk);

  // Sequence lengths and starts, then the longest-first order (ties: lower index):
  // for a longest-processing-time list (at most kMaxPersistLpt sequences) in LDS
  // arrays of their own, which consumer wave 0 reads while the first chain runs;
  // for more sequences in the V tile (scratch until the producers stage the first
  // chunk's V).  Chain 0 of bin b is the sequence of rank b either way.
  constexpr bool lpt = LPT;  // p.N <= kMaxPersistLpt
  int* plen = lpt ? sm.plen : reinterpret_cast<int*>(sm.V);
  int* pstart = lpt ? sm.pstart : plen + kMaxSortedSeqs;
  int* porder = lpt ? sm.porder : pstart + kMaxSortedSeqs;
  for (int s = tid; s < p.N; s += NTHREADS) {
    int64_t a = load_cu(p.cu_seqlens, p.cu_is_64, s), b = load_cu(p.cu_seqlens, p.cu_is_64, s + 1);
    a = a < 0 ? 0 : (a > p.T ? p.T : a);
    b = b < a ? a : (b > p.T ? p.T : b);
    plen[s] = int(b - a);
    pstart[s] = int(a);
  }
  // Blocks of T~, N and P that are never written per chunk are read as zeros.
  {
    const uint4 z = uint4{0u, 0u, 0u, 0u};
    for (int e = tid; e < C * TSTR / 8; e += NTHREADS) {
      reinterpret_cast<uint4*>(sm.P[0])[e] = z;
      reinterpret_cast<uint4*>(sm.P[1])[e] = z;
      reinterpret_cast<uint4*>(sm.Th[0])[e] = z;
      reinterpret_cast<uint4*>(sm.Th[1])[e] = z;
      reinterpret_cast<uint4*>(sm.Tl[0])[e] = z;
      reinterpret_cast<uint4*>(sm.Tl[1])[e] = z;
      if (e < NROWS * TSTR / 8) {
        reinterpret_cast<uint4*>(sm.Nh)[e] = z;
        reinterpret_cast<uint4*>(sm.Nl)[e] = z;
      }
    }
    if (tid < 16) sm.sync[tid] = 0;
    if (V::kHooks && tid == 0) {
      sm.spin_limit = p.spin_limit > 0 ? p.spin_limit : kSpinLimit;
      sm.aborts = p.aborts;
    }
    // Every list entry starts as an empty chain, so that no path (a wait for the list
    // that gave up included) reads one that was never written.
    for (int e = tid; e < kMaxPersistList; e += NTHREADS) {
      sm.pseq[e] = 0;
      sm.ps0[e] = 0;
      sm.ps1[e] = 0;
    }
    if (tid == 0) sm.pcount = 1;
  }
  __syncthreads();
  for (int s = tid; s < p.N; s += NTHREADS) {
    const int ls = plen[s];
    int r = 0;
    for (int j = 0; j < p.N; ++j) {
      const int lj = plen[j];
      r += (lj > ls) | ((lj == ls) & (j < s));
    }
    porder[r] = s;
    if (r == bin) {
      sm.pseq[0] = s;
      sm.ps0[0] = pstart[s];
      sm.ps1[0] = pstart[s] + ls;
    }
  }
  if constexpr (!lpt) {
    __syncthreads();  // porder complete
    // Many sequences: boustrophedon over the longest-first order.  Round j of B
    // ranks gives rank jB + b (j even) or jB + B - 1 - b (j odd) to bin b.
    const int cnt = p.N / nbins + (p.N % nbins > (p.N / nbins % 2 == 0 ? bin : nbins - 1 - bin));
    for (int j = 1 + tid; j < cnt; j += NTHREADS) {
      const int r = j * nbins + (j % 2 == 0 ? bin : nbins - 1 - bin);
      const int sj = porder[r];
      sm.pseq[j] = sj;
      sm.ps0[j] = pstart[sj];
      sm.ps1[j] = pstart[sj] + plen[sj];
    }
    if (tid == 0) {
      sm.pcount = cnt;
      sm.sync[kList] = 1;
    }
  }
  __syncthreads();  // chain 0 (with more sequences, the whole list), cleared LDS and counters

  if (wave >= NCW) {
    producer_loop<V>(sm, p, 0, 0, 0, h, hq, hk, 0, wave - NCW, lane0);
    return;
  }

  if (lpt && wave == 0) {
    // The rest of the list, while the producers prepare chain 0's first chunk:
    // longest-processing-time over the bins, longest first, each sequence onto the
    // least-loaded bin (cost 3 per chunk + 2 per sequence; ties to the lower bin;
    // the first B sequences go one per bin, in order).  Lane r holds the cost of the
    // sequence of rank r; lane b < B (at most 64) holds bin b's load.
    const int sr = lane0 < p.N ? porder[lane0] : 0;
    const int lr = lane0 < p.N ? plen[sr] : 0;
    const int cost_r = 3 * (lr / C + (lr % C != 0)) + 2;
    uint32_t load = lane0 < nbins ? 0u : 0xffffffffu;
    int cnt = 0;
    for (int r = 0; r < p.N; ++r) {
      const uint32_t m = wave_min(load);
      const int b = __builtin_ctzll(__ballot(load == m));
      if (lane0 == b) load += uint32_t(__builtin_amdgcn_readlane(cost_r, r));
      if (b == bin) {
        if (lane0 == r && cnt > 0) {
          sm.pseq[cnt] = sr;
          sm.ps0[cnt] = pstart[sr];
          sm.ps1[cnt] = pstart[sr] + lr;
        }
        ++cnt;
      }
    }
    if (lane0 == 0) sm.pcount = cnt;
    signal_count(sm, kList, lane0);
  }

  // Consumers: state rows v = VW*wave + vrow(vt, n16), cols k = 16*kt + 4g + i.
  const int g = lane0 >> 4, n16 = lane0 & 15;
  int nchains = 1;  // chain 0 now; the rest of the list once it is complete
  int u0 = 0;
  for (int k = 0; k < nchains; ++k) {
    const int seq = sm.pseq[k];
    const int64_t s0 = sm.ps0[k], s1 = sm.ps1[k];
    const int nchunks = int((s1 - s0 + C - 1) / C);
    const int64_t state_head = (int64_t(seq) * p.Hv + h) * D * D;
    f32x4 S[VT][8];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      const int v = VW * wave + vrow<VT>(vt, n16);
#pragma unroll
      for (int kt = 0; kt < 8; ++kt) {
        if (p.state) {
          const float4 x = *reinterpret_cast<const float4*>(p.state + state_head + int64_t(v) * D + 16 * kt + 4 * g);
          S[vt][kt] = f32x4{x.x, x.y, x.z, x.w};
        } else {
          S[vt][kt] = zero4();
        }
      }
    }
    if (nchunks > 0) {
      consumer_loop<V>(sm, p, s0, s1, nchunks, h, 0, wave, lane0, S, u0);
      u0 += nchunks;
    }
    // Final state (for an empty sequence: the initial state, or zeros).
    if (nchunks > 0 || p.state != p.new_state) {
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        const int v = VW * wave + vrow<VT>(vt, n16);
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) {
          const f32x4 x = S[vt][kt];
          *reinterpret_cast<float4*>(p.new_state + state_head + int64_t(v) * D + 16 * kt + 4 * g) =
              make_float4(x[0], x[1], x[2], x[3]);
        }
      }
    }
    if (k == 0) {
      wait_count<V::kHooks>(sm, kList, 1);  // the rest of the list
      nchains = chain_count(sm);
    }
  }
  if (aborted(sm)) {
    // A hand-off wait gave up: NaN over every output element and state element of
    // this wave's rows, in every chain of the workgroup.
    const int64_t vstride = int64_t(p.Hv) * D;
    for (int k = 0; k < nchains; ++k) {
      const int seq = sm.pseq[k];
      const int64_t s0 = sm.ps0[k], s1 = sm.ps1[k];
      uint16_t* obase = p.out + int64_t(h) * D + VW * wave + 8 * (lane0 >> 4);
      for (int64_t tok = s0 + n16; tok < s1; tok += 16)
        *reinterpret_cast<uint4*>(obase + tok * vstride) = uint4{kNaNx2, kNaNx2, kNaNx2, kNaNx2};
      const int64_t state_head = (int64_t(seq) * p.Hv + h) * D * D;
      const float nan = __builtin_nanf("");
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        const int v = VW * wave + vrow<VT>(vt, n16);
#pragma unroll
        for (int kt = 0; kt < 8; ++kt)
          *reinterpret_cast<float4*>(p.new_state + state_head + int64_t(v) * D + 16 * kt + 4 * g) =
              make_float4(nan, nan, nan, nan);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// State pass of the two-kernel path
// ---------------------------------------------------------------------------

// Rows 16 I + lane%16 of a chunk's K or Q slice (stride: bytes from token to token) as
// operands in kappa order, contraction blocks ks = 0 .. 3.  A lane loads 16 contiguous
// bytes a block (columns 32 ks + 8g .. +7, pieces 2g and 2g + 1 of four columns; rows past
// the chunk lie outside the buffer and read as zeros), and two row swaps deal the eight
// pieces of a row to its four lanes as kappa has them (lane g: pieces g and g + 4).  The
// order is that of the producers' LDS tiles, so the products are the same bit for bit.
struct RowFrags {
  u32x4 v[4];
  __device__ __forceinline__ void load(BufferRsrc r, int stride, int I, int lane) {
    const int off = (16 * I + (lane & 15)) * stride + 16 * (lane >> 4);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) v[ks] = __builtin_amdgcn_raw_buffer_load_b128(r, off + 64 * ks, 0, 0);
  }
  __device__ __forceinline__ void to_kappa() {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const auto x = __builtin_amdgcn_permlane16_swap(v[ks][i], v[ks][2 + i], false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(x[0], x[1], false, false);
        v[ks][i] = y[0];
        v[ks][2 + i] = y[1];
      }
  }
};

// LDS of the state pass.
struct __align__(16) StateSmem {
  uint16_t K[2][C * KSTR];               // K chunk [c][perm(k)], by chunk parity
  uint16_t T[2][8 * 2 * kTileUnits1];    // T~ hi, T~ lo: image fragments
  float gate[2][3 * C];                  // beta, e^gamma, e^{gamma_last - gamma}
  uint16_t V[2][C * 16];                 // V slice [token][state row]
  uint4 Y[4][64];                        // exchange: Y, 16-token blocks [block][lane]: hi, lo
  uint4 S[3][4][2][64];                  // exchange: state, 32-column blocks [block][hi, lo][lane]
  uint2 Vn[2][4][64];                    // v_new (hi parts), 16-token blocks [block][lane]
  int sync[16];                          // hand-off counters
  int seq;
};
// With testing hooks: as in PrefillSmem.
struct HookedStateSmem : StateSmem {
  int spin_limit;
  unsigned* aborts;
};
static_assert(sizeof(HookedStateSmem) <= 160 * 1024);

// Hand-offs of the state pass.  kAbort as in the other kernels.  "Loaded" and "output read"
// count by chunk parity: a helper wave may be a chunk ahead of another, and with one counter
// its signal could stand in for the other's.
enum StateCounter {
  kLoaded = 0,     // + parity: a helper wave stored its part of the chunk (4 a chunk)
  kChunkRead = 2,  // a consumer wave has read the chunk's buffers (4 a chunk)
  kStateIn = 3,        // a consumer wave stored its state columns (4 a chunk, 4 at start)
  kYIn = 5,        // a consumer wave stored its block of Y (4 a chunk)
  kVnewIn = 6,         // a consumer wave stored its block of v_new (4 a chunk)
  kOutRead = 7     // + parity: a helper wave has read the chunk's state and v_new (4 a chunk)
};
static_assert(kAbort == 4, "kAbort between the state pass's counters");

// What a helper thread moves of a chunk: K (four 16-byte units), T~ (three), gates and V.
struct StateLoad {
  u32x4 k[4], t[3], g, v;
};

constexpr int kStateLoaders = 256;  // helper threads (four waves)

// The helper waves keep off the chain whatever the state recurrence does not need.  Wave w
// * loads (its quarter of) K, T~, the gates and the V slice of chunk t into the LDS buffers
//   of parity t & 1 once the consumers are done with chunk t - 2.  The loads go two chunks
//   ahead (two register sets) and are unconditional (rows past the chunk lie outside the
//   buffer and read as zeros), so the compiler waits for exactly the older set;
// * forms and stores the output of the chunk's tokens 16w .. 16w + 15, from the chunk-start
//   state (hi parts) and v_new of the consumers' exchanges and its own Q rows and P
//   fragments, which no other wave reads: they go straight into registers.
// A wave that issues loads while the memory queue is full stalls (about 800 cycles a chunk);
// here that delays no consumer.
template <bool kHooks, class Smem>
__device__ __forceinline__ void state_helper(Smem& sm, const PrefillArgs& p, const u32x4* tiles, int64_t s0,
                                             int64_t s1, int nchunks, int h, int hq, int hk, int row0, int w,
                                             int lane0) {
  const int pt = 64 * w + lane0;
  const int ct = w;  // this wave's 16-token output block
  const int64_t vstride = int64_t(p.Hv) * D;
  const int kstr = p.Hk * D * 2, qstr = p.Hq * D * 2, vstr = p.Hv * D * 2;
  const int koff = (pt >> 4) * kstr + 16 * (pt & 15);
  const int voff = ((pt >> 1) & 63) * vstr + 16 * (pt & 1);
  const int goff = kTileUnits + min(pt, kGateUnits - 1);
  const int orow = (16 * ct + (lane0 & 15)) * int(vstride) + 4 * (lane0 >> 4);
  auto chunk_len = [&](int64_t cs) { return int(s1 - cs < C ? s1 - cs : C); };
  auto load = [&](int t, StateLoad& r) {
    const int64_t cs = s0 + int64_t(t) * C;
    const int clen = chunk_len(cs);
    const BufferRsrc kr = buffer_rsrc(const_cast<uint16_t*>(p.k) + (cs * p.Hk + hk) * D, uint32_t(clen - 1) * kstr + 2 * D);
    const BufferRsrc vr =
        buffer_rsrc(const_cast<uint16_t*>(p.v) + (cs * p.Hv + h) * D + row0, uint32_t(clen - 1) * vstr + 32);
    const u32x4* im = tiles + int64_t(t) * p.Hv * kTileImage;
#pragma unroll
    for (int it = 0; it < 4; ++it) r.k[it] = __builtin_amdgcn_raw_buffer_load_b128(kr, koff + 16 * it * kstr, 0, 0);
#pragma unroll
    for (int it = 0; it < 3; ++it) r.t[it] = im[pt + kStateLoaders * it];
    r.g = im[goff];
    r.v = __builtin_amdgcn_raw_buffer_load_b128(vr, voff, 0, 0);
  };
  auto stage = [&](int t, StateLoad& r, int lane) {
    const int b = t & 1;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int c = (pt >> 4) + 16 * it, sg = pt & 15;
      const int col0 = (8 * sg) & ~31, r0 = (8 * sg) & 31;
      *reinterpret_cast<uint2*>(sm.K[b] + kq_off(c, col0 + perm32(r0))) = uint2{r.k[it][0], r.k[it][1]};
      *reinterpret_cast<uint2*>(sm.K[b] + kq_off(c, col0 + perm32(r0 + 4))) = uint2{r.k[it][2], r.k[it][3]};
    }
#pragma unroll
    for (int it = 0; it < 3; ++it) *reinterpret_cast<u32x4*>(sm.T[b] + 8 * (pt + kStateLoaders * it)) = r.t[it];
    if (pt < kGateUnits) *reinterpret_cast<u32x4*>(sm.gate[b] + 4 * pt) = r.g;
    if (pt < 2 * C) *reinterpret_cast<u32x4*>(sm.V[b] + 8 * pt) = r.v;
    if (!kHooks || p.ready_chunks <= 0 || t < p.ready_chunks) signal_count(sm, kLoaded + b, lane);
  };
  // The output block's own operands: Q rows, P fragments and e^gamma of its tokens.
  RowFrags qf;
  u32x4 pf[2];
  float eo;
  auto load_out = [&](int t, int lane) {
    const int64_t cs = s0 + int64_t(t) * C;
    qf.load(buffer_rsrc(const_cast<uint16_t*>(p.q) + (cs * p.Hq + hq) * D, uint32_t(chunk_len(cs) - 1) * qstr + 2 * D),
            qstr, ct, lane);
    const u32x4* im = tiles + int64_t(t) * p.Hv * kTileImage;
    pf[0] = im[2 * kTileUnits1 + 64 * tile_frag(ct, 0) + lane];
    pf[1] = im[2 * kTileUnits1 + 64 * tile_frag(ct, ct >> 1) + lane];  // used by ct >= 2 only
    eo = reinterpret_cast<const float*>(im + kTileUnits)[C + 16 * ct + (lane & 15)];
  };
  // o^T = scale e^gamma (S Q^T) + v_new^T (scale P)^T of chunk t, tokens 16 ct .. +15.
  auto output = [&](int t, int sbuf, int lane) {
    wait_count<kHooks>(sm, kVnewIn, 4 * (t + 1));
    uint4 Sh[4];
    uint2 vn[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) Sh[ks] = sm.S[sbuf][ks][0][lane];
#pragma unroll
    for (int c = 0; c < 4; ++c) vn[c] = sm.Vn[t & 1][c][lane];
    signal_count(sm, kOutRead + (t & 1), lane);
    qf.to_kappa();
    f32x4 o = zero4();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) o = mfma(Sh[ks], __builtin_bit_cast(uint4, qf.v[ks]), o);
    o = o * (eo * p.scale);
    o = mfma(uint4{vn[0].x, vn[0].y, vn[1].x, vn[1].y}, __builtin_bit_cast(uint4, pf[0]), o);
    if (ct >= 2) o = mfma(uint4{vn[2].x, vn[2].y, vn[3].x, vn[3].y}, __builtin_bit_cast(uint4, pf[1]), o);
    // Rows at or past the chunk's end fall outside the buffer: the hardware drops their
    // stores (no per-lane branch).
    const int64_t cs = s0 + int64_t(t) * C;
    buffer_store8(u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])},
                  buffer_rsrc(p.out + cs * vstride + (int64_t(h) * D + row0),
                              uint32_t(chunk_len(cs)) * uint32_t(vstride) * 2u),
                  2 * orow);
  };
  StateLoad ra, rb;
  const int last = nchunks - 1;
  load(0, ra);
  load(min(1, last), rb);
  load_out(0, lane0);
  stage(0, ra, lane0);
  load(min(2, last), ra);
  if (last >= 1) stage(1, rb, lane0);
  load(min(3, last), rb);
  int sbuf = 0;  // t % 3
  auto tick = [&](int t, StateLoad& r) {
    int lane = lane0;
    asm volatile("" : "+v"(lane));
    // Chunk t + 2 first: the consumers take it sooner than they miss this output.
    if (t + 2 <= last) {
      wait_count<kHooks>(sm, kChunkRead, 4 * (t + 1));
      stage(t + 2, r, lane);
    }
    output(t, sbuf, lane);
    sbuf = sbuf == 2 ? 0 : sbuf + 1;
    load_out(min(t + 1, last), lane);
    load(min(t + 4, last), r);
  };
  for (int t = 0; t <= last; t += 2) {
    tick(t, ra);
    if (t + 1 <= last) tick(t + 1, rb);
  }
}

// The four consumer waves share the slice's 16 state rows: wave w keeps state columns
// 32w .. 32w + 31 in fp32, forms the rows of X = K S^T and Y of the chunk's tokens
// 16w .. 16w + 15, and updates its own columns.  Two LDS exchanges a chunk give every wave
// what the others formed: the four blocks of Y (for v_new, which every wave forms whole)
// and the bf16 hi/lo parts of the four column blocks of the state (for the next retrieve).
// Each value is produced by the same operations in the same order as in consumer_loop, so
// the results are those of the one-kernel path bit for bit.
//
// The chain of a chunk is LDS round trips and short dependent products (about 2.6k cycles,
// 1.3 us, a chunk), so every other operand is read where the wave computes or waits anyway:
// T~ behind the state, under the retrieve; the update's behind Y, under v_new; the next
// chunk's K rows, gates and V after the state is stored, while the other waves store theirs
// (under v_new they would hold up its first operands).  A wave splits its block of Y into
// bf16 hi and lo before the exchange, so that no wave splits all four.
//
// A wave rewrites its block of Y only after the wait for all four blocks of the state,
// which every wave signals after its last read of Y.  The state (three buffers) and v_new
// (two) are also read by the helpers, up to a chunk later.
//
// One 4,096-token sequence at 32 v-heads (256 workgroups, 64 chunks each), inputs from HBM,
// prep kernel included: 108 us a call; with K, Q, T~ and P all staged through the LDS and the
// outputs formed by the consumers 121.5; with the consumers loading their own K, Q and P
// rows into registers 152 (their loads stall behind the loaders').
template <bool kHooks, class Smem>
__device__ __forceinline__ void state_consumer(Smem& sm, const PrefillArgs& p, int64_t s0, int64_t s1, int nchunks,
                                               int wave, int lane0, f32x4 (&S)[2]) {
  const int ct = wave;  // this wave's 16-token block and 32-column block
  // K^T operand base of column blocks 2 ct, 2 ct + 1 (kt_bases with kt / 2 = ct).
  int ktb;
  {
    const int j = lane0 & 15, rl = 4 * (lane0 >> 4) + (j >> 2), sl = kq_sigma(rl);
    ktb = rl * KSTR + 8 * ((j & 3) ^ (sl & 3)) + 32 * (ct ^ (sl >> 2));
  }
  // What the retrieve and Y of a chunk take besides the state, read a chunk ahead.
  uint4 kf[4];
  f32x4 b4, e4;
  uint2 vv;
  auto read_ahead = [&](int t, int lane) {
    const int b = t & 1, g = lane >> 4, n16 = lane & 15;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) kf[ks] = frag_kq(sm.K[b], 16 * ct, ks, lane);
    b4 = ld4(sm.gate[b] + 16 * ct + 4 * g);
    e4 = ld4(sm.gate[b] + C + 16 * ct + 4 * g);
    vv = read_tr(sm.V[b] + (16 * ct + 4 * g + (n16 >> 2)) * 16 + 4 * (n16 & 3));
  };
  auto put_state = [&](int sbuf, int lane) {
    uint4 Sh, Sl;
    split_pack(S[0], S[1], Sh, Sl);
    sm.S[sbuf][ct][0][lane] = Sh;
    sm.S[sbuf][ct][1][lane] = Sl;
    signal_count(sm, kStateIn, lane);
  };
  put_state(0, lane0);
  wait_count<kHooks>(sm, kLoaded, 4);
  read_ahead(0, lane0);
  int sbuf = 0;  // t % 3
  for (int t = 0; t < nchunks; ++t) {
    int lane = lane0;
    asm volatile("" : "+v"(lane));
    const int g = lane >> 4;
    const int64_t cs = s0 + int64_t(t) * C;
    const int clen = int(s1 - cs < C ? s1 - cs : C);
    const int b = t & 1;
    // The chunk-start state; the next chunk's buffers looked at in the same read (the last
    // chunk looks at its own).
    const int tn = min(t + 1, nchunks - 1);
    const bool loaded = wait_count_peek<kHooks>(sm, kStateIn, 4 * (t + 1), kLoaded + (tn & 1), 4 * ((tn >> 1) + 1));
    uint4 Sh[4], Sl[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      Sh[ks] = sm.S[sbuf][ks][0][lane];
      Sl[ks] = sm.S[sbuf][ks][1][lane];
    }
    __builtin_amdgcn_sched_barrier(0);
    uint4 thf[kTileFrags], tlf[kTileFrags];  // T~
#pragma unroll
    for (int i = 0; i < kTileFrags; ++i) {
      thf[i] = *reinterpret_cast<const uint4*>(sm.T[b] + 8 * (64 * i + lane));
      tlf[i] = *reinterpret_cast<const uint4*>(sm.T[b] + 8 * (kTileUnits1 + 64 * i + lane));
    }
    __builtin_amdgcn_sched_barrier(0);

    // 1: block ct of X = K S^T; Y for rows c = 16ct + 4g + i, as consumer_loop.
    f32x4 xk = zero4();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      xk = mfma(kf[ks], Sh[ks], xk);
      xk = mfma(kf[ks], Sl[ks], xk);
    }
    {
      const float vf[4] = {bf16lo_f32(vv.x), bf16hi_f32(vv.x), bf16lo_f32(vv.y), bf16hi_f32(vv.y)};
#pragma unroll
      for (int i = 0; i < 4; ++i) xk[i] = b4[i] * (vf[i] - e4[i] * xk[i]);
    }
    {
      uint2 hi, lo;
      split4(xk, hi, lo);
      sm.Y[ct][lane] = uint4{hi.x, hi.y, lo.x, lo.y};
    }
    signal_count(sm, kYIn, lane);
    // All of Y; the helpers done with the v_new (of chunk t - 2) and the state (before it)
    // whose buffers this chunk rewrites, looked at in the same read.
    const bool out_read = wait_count_peek<kHooks>(sm, kYIn, 4 * (t + 1), kOutRead + b, 4 * (t >> 1));
    uint4 Y[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) Y[c] = sm.Y[c][lane];
    __builtin_amdgcn_sched_barrier(0);
    // The update's operands: its decays and K^T (columns 32ct .. +31).
    const float dlast = sm.gate[b][C + clen - 1];
    f32x4 ed[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) ed[c] = ld4(sm.gate[b] + 2 * C + 16 * c + 4 * g);
    uint4 kt[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int js = 0; js < 2; ++js) {
        const uint16_t* kp = sm.K[b] + ktb + 32 * js * KSTR + 4 * j;
        const uint2 k0 = read_tr(kp), k1 = read_tr(kp + 16 * KSTR);
        kt[j][js] = uint4{k0.x, k0.y, k1.x, k1.y};
      }
    signal_count(sm, kChunkRead, lane);  // buffers of this chunk no longer read
    __builtin_amdgcn_sched_barrier(0);

    // 2: v_new = T~ Y, all 64 rows; this wave's block of it (hi parts) to the helpers.
    uint4 Yh[2], Yl[2];
#pragma unroll
    for (int js = 0; js < 2; ++js) {
      Yh[js] = uint4{Y[2 * js].x, Y[2 * js].y, Y[2 * js + 1].x, Y[2 * js + 1].y};
      Yl[js] = uint4{Y[2 * js].z, Y[2 * js].w, Y[2 * js + 1].z, Y[2 * js + 1].w};
    }
    f32x4 Vn[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      Vn[c] = zero4();
#pragma unroll
      for (int js = 0; js <= (c >> 1); ++js) {
        const uint4 th = thf[tile_frag(c, js)], tl = tlf[tile_frag(c, js)];
        Vn[c] = mfma(th, Yh[js], Vn[c]);
        Vn[c] = mfma(th, Yl[js], Vn[c]);
        Vn[c] = mfma(tl, Yh[js], Vn[c]);
      }
    }
    if (!out_read) wait_count<kHooks>(sm, kOutRead + b, 4 * (t >> 1));

    // 3: columns 32ct .. 32ct + 31 of S = e^{gamma_last} S + sum_c K[c]^T (d_c v_new[c]).
    uint4 Uh[2], Ul[2];
#pragma unroll
    for (int js = 0; js < 2; ++js) split_pack(Vn[2 * js] * ed[2 * js], Vn[2 * js + 1] * ed[2 * js + 1], Uh[js], Ul[js]);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      S[j] = S[j] * dlast;
#pragma unroll
      for (int js = 0; js < 2; ++js) {
        S[j] = mfma(kt[j][js], Uh[js], S[j]);
        S[j] = mfma(kt[j][js], Ul[js], S[j]);
      }
    }
    sbuf = sbuf == 2 ? 0 : sbuf + 1;
    put_state(sbuf, lane);
    const f32x4 v = ct == 0 ? Vn[0] : ct == 1 ? Vn[1] : ct == 2 ? Vn[2] : Vn[3];
    sm.Vn[b][ct][lane] = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    signal_count(sm, kVnewIn, lane);
    if (t + 1 < nchunks) {
      if (!loaded) wait_count<kHooks>(sm, kLoaded + (tn & 1), 4 * ((tn >> 1) + 1));
      read_ahead(tn, lane);
    }
  }
}

// Workgroup b handles slice f (16 state rows) of chain `chain` (rank-major, v-head minor),
// placed as in gdn_prefill_kernel with F = 8: the slices of a GQA pair of chains share an
// XCD.  Waves 0-3 are consumers, 4-7 helpers.
constexpr int kStateSlices = 8;
template <bool HOOKS>
__global__ __launch_bounds__(512) void gdn_prefill_state_kernel(PrefillArgs p) {
  constexpr int F = kStateSlices;
  __shared__ std::conditional_t<HOOKS, HookedStateSmem, StateSmem> sm;
  const int tid = threadIdx.x;
  const int lane0 = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bid = blockIdx.x;
  const int chain = (bid / (16 * F)) * 16 + 2 * (bid % 8) + (bid / 8) % (2 * F) / F;
  const int row0 = ((bid / 8) % F) * 16;
  if (chain >= p.N * p.Hv) return;  // padding of the last group of 16 chains (workgroup-uniform)
  const int h = chain % p.Hv;
  const int seq = pick_sequence<512>(reinterpret_cast<int*>(sm.K), &sm.seq, p, chain / p.Hv, tid);
  const int hq = h / (p.Hv / p.Hq);
  const int hk = h / (p.Hv / p.Hk);
  const SeqRange sr = seq_range(p, seq);
  const int64_t s0 = sr.s0, s1 = sr.s1;
  const int nchunks = int((s1 - s0 + C - 1) / C);
  if (tid < 16) sm.sync[tid] = 0;
  if constexpr (HOOKS) {
    if (tid == 0) {
      sm.spin_limit = p.spin_limit > 0 ? p.spin_limit : kSpinLimit;
      sm.aborts = p.aborts;
    }
  }
  __syncthreads();  // counters cleared; pick_sequence's scratch read
  const u32x4* tiles =
      reinterpret_cast<const u32x4*>(p.tiles) + (int64_t(chunks_before(p, seq, lane0)) * p.Hv + h) * kTileImage;

  if (wave >= 4) {
    if (nchunks > 0) {
      state_helper<HOOKS>(sm, p, tiles, s0, s1, nchunks, h, hq, hk, row0, wave - 4, lane0);
      if (aborted(sm)) {
        // A hand-off wait gave up: NaN over the slice's outputs (wave w: tokens
        // s0 + 16 (4m + w) + lane % 16).
        const int64_t vstride = int64_t(p.Hv) * D;
        uint16_t* obase = p.out + int64_t(h) * D + row0 + 4 * (lane0 >> 4);
        for (int64_t tok = s0 + 16 * (wave - 4) + (lane0 & 15); tok < s1; tok += 64)
          *reinterpret_cast<uint2*>(obase + tok * vstride) = uint2{kNaNx2, kNaNx2};
      }
    }
    return;
  }

  // Wave w holds column blocks 2w and 2w + 1 (cols k = 16 kt + 4g + i) of the slice's
  // rows v = row0 + n16.
  const int g = lane0 >> 4, n16 = lane0 & 15;
  const int64_t srow = (int64_t(seq) * p.Hv + h) * D * D + int64_t(row0 + n16) * D + 32 * wave + 4 * g;
  f32x4 S[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    S[j] = zero4();
    if (p.state) S[j] = ld4(p.state + srow + 16 * j);
  }
  if (nchunks > 0) {
    state_consumer<HOOKS>(sm, p, s0, s1, nchunks, wave, lane0, S);
    if (aborted(sm)) {  // a hand-off wait gave up: NaN over the slice's state
      const float nan = __builtin_nanf("");
      S[0] = S[1] = f32x4{nan, nan, nan, nan};
    }
  }
  if (nchunks > 0 || p.state != p.new_state) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      *reinterpret_cast<float4*>(p.new_state + srow + 16 * j) = make_float4(S[j][0], S[j][1], S[j][2], S[j][3]);
  }
}

// ---------------------------------------------------------------------------
// Prep kernel of the two-kernel path: T~, P and the gates of every chunk-head, one
// wave each.
// ---------------------------------------------------------------------------

__device__ __forceinline__ f32x4 row_product(const RowFrags& a, const RowFrags& b) {
  f32x4 acc = zero4();
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    acc = mfma(__builtin_bit_cast(uint4, a.v[ks]), __builtin_bit_cast(uint4, b.v[ks]), acc);
  return acc;
}

// Four rows 4g .. +3 of column lane%16 of a 16x16 block stored column-major (a 16x16x16 B
// operand), and row lane%16, columns 4g .. +3 (an A operand), by a transpose read.
__device__ __forceinline__ uint2 block_rows_of_col(const uint16_t* blk, int lane) {
  return *reinterpret_cast<const uint2*>(blk + 16 * (lane & 15) + 4 * (lane >> 4));
}
__device__ __forceinline__ uint2 block_cols_of_row(const uint16_t* blk, int lane) {
  return read_tr(blk + 16 * (4 * (lane >> 4) + ((lane & 15) >> 2)) + 4 * (lane & 3));
}

// A block X (accumulator layout), split, as an A operand, through the wave's LDS.
__device__ __forceinline__ void put_block(uint16_t (&blk)[2][256], const f32x4& X, int lane) {
  uint2 hi, lo;
  split4(X, hi, lo);
  *reinterpret_cast<uint2*>(blk[0] + 16 * (lane & 15) + 4 * (lane >> 4)) = hi;
  *reinterpret_cast<uint2*>(blk[1] + 16 * (lane & 15) + 4 * (lane >> 4)) = lo;
}
__device__ __forceinline__ Pair2 get_block(const uint16_t (&blk)[2][256], int lane) {
  return Pair2{block_cols_of_row(blk[0], lane), block_cols_of_row(blk[1], lane)};
}

// Wave item (chunk number, v-head) prepares that chunk-head: the same values, from the same
// operations in the same order, as the producers of the one-kernel path, but without their
// hand-offs.  K and Q rows go from global memory into the operands, the N tiles stay in
// registers (an N tile's accumulator layout is the A operand the off-diagonal solve takes),
// the tiles (I, J) of N and P share their decays, and every fragment of the image leaves
// the registers as a linear 16-byte store.  A chunk-head is a chain of dependent steps
// (about 9k cycles of arithmetic and 5k of first loads), so a small batch takes that long
// whatever its size (32 v-heads, inputs cached: 640 tokens, 320 chunk-heads, 8.9 us, 1,024
// tokens 9.4), and what counts is how many are in flight: 12 waves a CU, no barriers.
// Larger batches move towards the memory's pace: 2,048 tokens 14.2, 4,096 22.2, 8,192 37.0,
// 12,288 50.8, the last 145 MB of K, Q and images at 5.1 TB/s, where a device copy reaches
// 5.3 (a sixth of the tile bytes are the zeros of fragments (0, 0) and (2, 1)).  A
// workgroup of four waves per run of chunks, handing over through the LDS (two workgroups a
// CU), took 26.9 us at 4,096 tokens with inputs from HBM against 20.6, and about 80 at
// 12,288 against 51.7.
constexpr int kPrepWaves = 2;
__global__ __launch_bounds__(64 * kPrepWaves, 2) void gdn_prefill_prep_kernel(PrefillArgs p) {
  __shared__ PrepSmem smem[kPrepWaves];
  const int lane0 = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  PrepSmem& sm = smem[wave];
  // v-heads 2j and 2j + 1 of a chunk, which read the same K and Q, share a workgroup.
  const int item = int(blockIdx.x) * kPrepWaves + wave;
  const int h = item % p.Hv;
  const int hq = h / (p.Hv / p.Hq);
  const int hk = h / (p.Hv / p.Hk);
  const float neg_decay = -expf(p.A_log[h]), dt_bias = p.dt_bias[h];
  // One pass, except for malformed offsets whose sequences overlap: their chunks can
  // exceed prep_slots.  (Items past the last chunk-head have slot >= prep_slots.)
  for (int slot = item / p.Hv;; slot += p.prep_slots) {
    int lane = lane0;  // opaque, so that lane-dependent addresses are not hoisted and spilled
    asm volatile("" : "+v"(lane));
    const int g = lane >> 4, n16 = lane & 15;
    const ChunkAt c = find_chunk(p, slot, lane);
    if (c.clen <= 0) break;
    const int64_t cs = c.start;
    const int clen = c.clen;
    u32x4* image = reinterpret_cast<u32x4*>(p.tiles) + (int64_t(slot) * p.Hv + h) * kTileImage;
    const int kstr = p.Hk * D * 2, qstr = p.Hq * D * 2;
    const BufferRsrc kr = buffer_rsrc(const_cast<uint16_t*>(p.k) + (cs * p.Hk + hk) * D, uint32_t(clen - 1) * kstr + 2 * D);
    const BufferRsrc qr = buffer_rsrc(const_cast<uint16_t*>(p.q) + (cs * p.Hq + hq) * D, uint32_t(clen - 1) * qstr + 2 * D);
    ProducerPrefetch f;
    {
      const int row = lane < clen ? lane : clen - 1;
      f.a = (p.a + cs * p.Hv + h)[row * p.Hv];
      f.b = (p.b + cs * p.Hv + h)[row * p.Hv];
    }
    // The loads go out two row blocks ahead of their use: a wave that issued all of them
    // at once would wait for the memory queue, and all waves for the same memory, before
    // any of them computes.
    RowFrags k[4], q[4];
    auto load_block = [&](int I) {
      k[I].load(kr, kstr, I, lane);
      q[I].load(qr, qstr, I, lane);
      __builtin_amdgcn_sched_barrier(0);
    };
    load_block(0);
    load_block(1);
    {
      const ChunkGates gts = chunk_gates(f, lane, clen, neg_decay, dt_bias);
      sm.gam[lane] = gts.gam;
      sm.gaml[lane] = gts.gaml;
      sm.bet[lane] = gts.bet;
      float* gi = reinterpret_cast<float*>(image + kTileUnits);
      gi[lane] = gts.bet;
      gi[C + lane] = gts.eg;
      gi[2 * C + lane] = gts.dd;
    }
    wave_lds_sync();

    // Tiles (I, J), J <= I: decay e^{gamma_r - gamma_c} for r = 16I + n16, c = 16J + 4g + i;
    // N[r][c] from k_c . k_r (off-diagonal: an A operand; diagonal: fp32, column-major) and
    // P[r][c] from k_c . q_r (c <= r), with the output scale folded in.
    Pair2 n[4][3];
#pragma unroll
    for (int I = 0; I < 4; ++I) {
      if (I < 2) load_block(I + 2);
      k[I].to_kappa();
      q[I].to_kappa();
      const int r = 16 * I + n16;
      const float gr = sm.gam[r], grl = sm.gaml[r], br = sm.bet[r];
      uint2 pt[4] = {uint2{0u, 0u}, uint2{0u, 0u}, uint2{0u, 0u}, uint2{0u, 0u}};
#pragma unroll
      for (int J = 0; J <= I; ++J) {
        const f32x4 an = row_product(k[J], k[I]), ap = row_product(k[J], q[I]);
        const f32x4 gcv = ld4(sm.gam + 16 * J + 4 * g), gcl = ld4(sm.gaml + 16 * J + 4 * g);
        f32x4 e, x;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          e[i] = exp2_le0(fminf(gamma_diff(gr, grl, gcv[i], gcl[i]), 0.f));
          x[i] = br * e[i] * an[i];
        }
        if (J < I) {
          split4(x, n[I][J < 3 ? J : 0].h, n[I][J < 3 ? J : 0].l);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) sm.Nd[I * NDB + (4 * g + i) * 16 + n16] = x[i];
        }
        float pv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float y = e[i] * (ap[i] * p.scale);
          pv[i] = J < I || 4 * g + i <= n16 ? y : 0.f;
        }
        pt[J] = uint2{pack_bf16x2(pv[0], pv[1]), pack_bf16x2(pv[2], pv[3])};
      }
#pragma unroll
      for (int js = 0; js <= I / 2; ++js)
        image[2 * kTileUnits1 + 64 * tile_frag(I, js) + lane] =
            u32x4{pt[2 * js].x, pt[2 * js].y, pt[2 * js + 1].x, pt[2 * js + 1].y};
    }
    wave_lds_sync();

    // Diagonal blocks of T~: lane (r, j) forms column j of block r.
    {
      float x[16];
      diag_columns(sm.Nd, x, lane);
      uint2 hi[4], lo[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) split4(f32x4{x[4 * m], x[4 * m + 1], x[4 * m + 2], x[4 * m + 3]}, hi[m], lo[m]);
      uint4* dh = reinterpret_cast<uint4*>(sm.D[0] + 16 * lane);
      uint4* dl = reinterpret_cast<uint4*>(sm.D[1] + 16 * lane);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        dh[m] = uint4{hi[2 * m].x, hi[2 * m].y, hi[2 * m + 1].x, hi[2 * m + 1].y};
        dl[m] = uint4{lo[2 * m].x, lo[2 * m].y, lo[2 * m + 1].x, lo[2 * m + 1].y};
      }
    }
    wave_lds_sync();

    // Off-diagonal blocks (the products and order of offdiag_right and offdiag_left).
    Pair2 a[4], d[3];  // D_I as A operands, D_0 .. D_2 as B operands
#pragma unroll
    for (int I = 0; I < 4; ++I) {
      a[I] = Pair2{block_cols_of_row(sm.D[0] + 256 * I, lane), block_cols_of_row(sm.D[1] + 256 * I, lane)};
      if (I < 3) d[I] = Pair2{block_rows_of_col(sm.D[0] + 256 * I, lane), block_rows_of_col(sm.D[1] + 256 * I, lane)};
    }
    const f32x4 g32 = mul3_16(zero4(), n[3][2], d[2]);
    const f32x4 g10 = mul3_16(zero4(), n[1][0], d[0]);
    const f32x4 m21 = mul3_16(zero4(), n[2][1], d[1]);
    const f32x4 m31 = mul3_16(zero4(), n[3][1], d[1]);
    const f32x4 p20 = mul3_16(zero4(), n[2][0], d[0]);
    const f32x4 p30 = mul3_16(zero4(), n[3][0], d[0]);
    const Pair2 ng32 = acc_b(-g32), ng10 = acc_b(-g10), nm21 = acc_b(-m21), nm31 = acc_b(-m31);
    put_block(sm.X[5], mul3_16(zero4(), a[3], ng32), lane);  // X32
    const f32x4 x10 = mul3_16(zero4(), a[1], ng10);
    const Pair2 x32t = acc_b(mul3_16(zero4(), ng32, a[3]));
    put_block(sm.X[0], x10, lane);  // X10
    const Pair2 b10 = acc_b(x10);
    const Pair2 nm20 = acc_b(-mul3_16(p20, n[2][1], b10));
    const Pair2 nm30 = acc_b(-mul3_16(p30, n[3][1], b10));
    put_block(sm.X[2], mul3_16(zero4(), a[2], nm21), lane);                                  // X21
    put_block(sm.X[4], mul3_16(mul3_16(zero4(), x32t, nm21), a[3], nm31), lane);             // X31
    put_block(sm.X[1], mul3_16(zero4(), a[2], nm20), lane);                                  // X20
    wave_lds_sync();
    const Pair2 x32 = get_block(sm.X[5], lane);
    put_block(sm.X[3], mul3_16(mul3_16(zero4(), a[3], nm30), x32, nm20), lane);              // X30
    wave_lds_sync();
    const Pair2 t10 = get_block(sm.X[0], lane), t20 = get_block(sm.X[1], lane), t21 = get_block(sm.X[2], lane),
                t30 = get_block(sm.X[3], lane), t31 = get_block(sm.X[4], lane);
    const Pair2 zero = {uint2{0u, 0u}, uint2{0u, 0u}};
    auto store_frag = [&](int frag, const Pair2& left, const Pair2& right) {
      image[64 * frag + lane] = u32x4{left.h.x, left.h.y, right.h.x, right.h.y};
      image[kTileUnits1 + 64 * frag + lane] = u32x4{left.l.x, left.l.y, right.l.x, right.l.y};
    };
    store_frag(tile_frag(0, 0), a[0], zero);
    store_frag(tile_frag(1, 0), t10, a[1]);
    store_frag(tile_frag(2, 0), t20, t21);
    store_frag(tile_frag(2, 1), a[2], zero);
    store_frag(tile_frag(3, 0), t30, t31);
    store_frag(tile_frag(3, 1), x32, a[3]);
    if (slot + p.prep_slots >= c.total) break;
    wave_lds_sync();
  }
}

// `done`, if not null, is recorded by the launch itself when the kernel completes
// (the kernel's own completion signal; no separate marker in the stream).
template <class V>
hipError_t launch_variant(const PrefillArgs& a, hipStream_t stream, hipEvent_t done = nullptr) {
  const int64_t chains = int64_t(a.N) * a.Hv;
  const int64_t grid = (chains + 15) / 16 * 16 * V::F;
  if (done != nullptr) {
    hipExtLaunchKernelGGL(gdn_prefill_kernel<V>, dim3(unsigned(grid)), dim3(V::NTHREADS), 0, stream, nullptr, done, 0,
                          a);
  } else {
    hipLaunchKernelGGL(gdn_prefill_kernel<V>, dim3(unsigned(grid)), dim3(V::NTHREADS), 0, stream, a);
  }
  return hipGetLastError();
}

int device_cus();

// Batches of more chains than CUs run persistently where they can: a workgroup per
// CU, Hv dividing the CUs into B <= 64 bins, at most kMaxSortedSeqs sequences and
// kMaxPersistList per bin.
bool persistent_batch(const PrefillArgs& a) {
  const int cus = device_cus();
  if (cus % a.Hv != 0 || cus / a.Hv > 64 || a.N > kMaxSortedSeqs || int64_t(a.N) * a.Hv <= cus) return false;
  const int bins = cus / a.Hv;
  return (a.N + bins - 1) / bins <= kMaxPersistList;
}

template <class V>
hipError_t launch_persistent(const PrefillArgs& a, hipStream_t stream) {
  if (a.N <= kMaxPersistLpt) {
    hipLaunchKernelGGL((gdn_prefill_persistent_kernel<V, true>), dim3(unsigned(device_cus())), dim3(V::NTHREADS), 0,
                       stream, a);
  } else {
    hipLaunchKernelGGL((gdn_prefill_persistent_kernel<V, false>), dim3(unsigned(device_cus())), dim3(V::NTHREADS), 0,
                       stream, a);
  }
  return hipGetLastError();
}

// Compute units of the current device (queried once per device).
int device_cus() {
  static std::atomic<int> cus[64];  // 0 until queried; racing first queries store the same value
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cus[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

}  // namespace

// Scratch of gdn_prefill_no_alloc: the chunk images of the two-kernel path, for
// callers that cannot allocate.  Each device that loads the library holds its own
// copy until the process ends; every call on a device shares it.
static __device__ __align__(256) uint8_t scratch[kPrefillScratchBytes];

// Scratch of the drop-in gdn_prefill's two-kernel path (long sequences, below):
// its own array, so that no call of gdn_prefill_no_alloc, captured or not, shares it.
static __device__ __align__(256) uint8_t dropin_scratch[kPrefillDropinScratchBytes];

namespace {
constexpr int kMaxDevices = 64;

// Per device and scratch array: the array's device address (looked up once, with
// the device current: in host code the array's name is a host-side stand-in), the
// event that follows the last launch using it, and the lock that orders the
// check-launch-record sequence between host threads.  Created on first use and
// kept until the process ends, like the array itself.  The stream (and thread, for the
// per-thread default stream) of the last launch only decides whether a batch that yields
// takes the array: what keeps launches apart is the event.
struct OrderedScratch {
  std::mutex lock;
  void* addr = nullptr;
  hipEvent_t done = nullptr;
  bool used = false;
  hipStream_t stream = nullptr;
  std::thread::id thread;
};
OrderedScratch g_dropin[kMaxDevices];
OrderedScratch g_no_alloc[kMaxDevices];

hipError_t launch_two_kernels(const PrefillArgs& a, hipStream_t stream, int64_t slots, hipEvent_t done);

// The array's entry for the current device.
hipError_t ordered_scratch(OrderedScratch* table, OrderedScratch** entry) {
  int dev = 0;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  *entry = table + dev;
  return hipSuccess;
}

// Whether another stream's launch holds the array (its lock held by the caller): a launch
// on `stream` would wait for it.
bool held_by_another(const OrderedScratch& d, hipStream_t stream) {
  if (!d.used) return false;
  if (d.stream == stream && (stream != hipStreamPerThread || d.thread == std::this_thread::get_id())) return false;
  // (An event query is not allowed while any thread captures a graph in the global mode,
  // unless the querying thread has relaxed its own.)
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return true;
  const hipError_t q = hipEventQuery(d.done);
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  if (q != hipSuccess) (void)hipGetLastError();  // not ready
  return q != hipSuccess;
}

// Launches the two-kernel path of `a` with its chunk images in the scratch array
// `symbol`, ordered after the previous launch that used the array on this device:
// the stream waits for that launch's event, and the state pass records the event
// again as it completes.  If the launch fails after the prep kernel was enqueued,
// the event is recorded behind it all the same, so the next launch still waits for
// the orphaned kernel.  With `yields`, runs launch_prefill instead if the array is held
// by another stream's launch.
hipError_t launch_ordered(const PrefillArgs& a, hipStream_t stream, OrderedScratch* table, const void* symbol,
                          int64_t bytes, bool yields) {
  OrderedScratch* entry = nullptr;
  hipError_t e = ordered_scratch(table, &entry);
  if (e != hipSuccess) return e;
  OrderedScratch& d = *entry;
  std::unique_lock<std::mutex> guard(d.lock);
  if (yields && held_by_another(d, stream)) {
    guard.unlock();
    return launch_prefill(a, stream);
  }
  if (d.addr == nullptr) {
    e = hipGetSymbolAddress(&d.addr, symbol);
    if (e != hipSuccess) return e;
  }
  if (d.done == nullptr) {
    e = hipEventCreate(&d.done);
    if (e != hipSuccess) return e;
  }
  if (d.used) {
    e = hipStreamWaitEvent(stream, d.done, 0);
    if (e != hipSuccess) return e;
  }
  PrefillArgs b = a;
  b.tiles = static_cast<uint16_t*>(d.addr);
  // The (last) state pass records `done` as it completes.
  e = launch_two_kernels(b, stream, bytes / (int64_t(a.Hv) * kTileImage * 16), d.done);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    (void)hipEventRecord(d.done, stream);
  }
  d.used = true;
  d.stream = stream;
  d.thread = std::this_thread::get_id();
  return e;
}

bool stream_capturing(hipStream_t stream, hipError_t* err) {
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  *err = hipStreamIsCapturing(stream, &capture);
  return *err == hipSuccess && capture != hipStreamCaptureStatusNone;
}
}  // namespace

// The device address of `scratch` on the current device, looked up once per
// device (with that device current) and kept.  In host code `scratch` names a
// host-side stand-in, so kernels and copies must use this address instead.
hipError_t prefill_scratch(void** ptr) {
  static std::atomic<void*> addr[kMaxDevices];  // null until looked up; racing lookups store the same value
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  void* p = addr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    addr[dev].store(p, std::memory_order_release);
  }
  *ptr = p;
  return hipSuccess;
}

int64_t prefill_static_device_bytes() {
  return int64_t(sizeof(scratch)) + int64_t(sizeof(dropin_scratch)) + int64_t(sizeof(gdn_prefill_giveup_count));
}

namespace {
int split_factor(int64_t chains);

// Windows of the two-kernel path with room for `slots` chunk images a v-head (at least N):
// their number and the chunks of each sequence that one covers.  If the chunks that any
// offsets can give do not fit (one or two sequences cannot overlap: at most ceil(T / C) + N
// - 1; more, if malformed, can: N ceil(T / C)), the batch runs in windows of equally many
// chunks of every sequence.
struct Windows {
  int64_t count, chunks;
};
Windows plan_windows(int64_t N, int64_t T, int64_t slots) {
  const int64_t tc = (T + C - 1) / C;
  const int64_t most = N <= 2 ? tc + N - 1 : N * tc;  // chunks any offsets can give
  const int64_t fit = most <= slots ? tc : slots / N;  // chunks of a sequence a window
  const int64_t count = (tc + fit - 1) / fit;
  return Windows{count, (tc + count - 1) / count};
}
}  // namespace

// How the drop-in runs a batch.  The host sees N and T, not the lengths, so the line between
// one kernel and two is drawn by the average length, where equal lengths gain nothing yet
// (ragged batches, which end with their longest chain, gain from there on).  One kernel
// against two in the drop-in's scratch, us:
//  * split 8 ways, from 640 tokens: one sequence at 32 v-heads 512 tokens 25.0 / 25.7, 640
//    29.8 / 28.5, 768 34.5 / 31.2; two of 640 at 16 v-heads 30.4 / 29.8;
//  * split 4 ways, from 1,024: [640, 640] 35.5 / 39.7, [900, 900] 49.1 / 48.9, [2048, 2048]
//    111 / 86.0;
//  * split 2 ways, from 1,024 where three eighths of the CUs or fewer have a chain: the
//    state pass saves about a third of a chunk of the longest chain, the prep kernel adds
//    10 us per 1,000 chunk-heads.  96 chains: [1024] x 3 63.6 / 61.5, [100, 3000, 900] 169.5 /
//    127.6, [768] x 3 49.6 / 49.6; 128 chains: [1024] x 4 67.7 / 69.5, [2048] x 4 126.8 / 132.0
//    (but [1000, 1500, 300, 1307] 93.0 / 86.6).
//
// Launches in the scratch run one after another, whatever their streams.  Below 1,024 tokens,
// and split 2 ways, that costs calls on several streams more than two kernels give them, so
// those batches yield: one kernel while another stream's launch holds the scratch.  A call
// on each of several streams, us, one kernel / two kernels in turn / yielding: [700] at 16
// v-heads on two streams 39.5 / 72 / 34, at 32 62 / 77 / 61, at 8 on four 79 / 141 / 80;
// [1024] x 3 at 32 on two 94.5 / 125 / 89; [4096, 4096] at 48 356 / 431 / 348.
//
// One or two sequences run in windows if their images do not fit the scratch; for more, as
// offsets that overlap have to fit too (N ceil(T / C) images a v-head), windows would mostly
// be empty (in twice the scratch, twelve sequences of 1,024 at 8 v-heads, two windows, the
// second of them empty: 63.8 / 69.7).  Windows hold the scratch for long, so they are for
// batches that leave other streams little room anyway, with a workgroup on three quarters of
// the CUs: a call on each of two streams, one kernel / windows, [16384] at 32 v-heads 1,196 /
// 845, at 24 v-heads 20,000 tokens 1,464 / 988; but at 16 v-heads 30,000 tokens 1,099 /
// 1,353, at 8 60,000 2,204 / 2,549, and split 2 ways [8192, 8192] at 48 706 / 903.
PrefillRoute dropin_route(int N, int64_t T, int Hv) {
  const PrefillRoute one_kernel = {0, false};
  if (N <= 0 || T <= 0) return one_kernel;
  const int64_t chains = int64_t(N) * Hv, cus = device_cus();
  const int F = split_factor(chains);
  if (F < 2 || (F == 2 && 8 * chains > 3 * cus)) return one_kernel;
  if (T < (F == 8 ? kDropinTwoKernelTokens8 : kDropinTwoKernelTokens) * N) return one_kernel;
  PrefillRoute r = {1, F == 2 || T < kDropinTwoKernelTokens * N};
  if (chains * ((T + C - 1) / C) * kTileImage * 16 > kPrefillDropinScratchBytes) {
    if (N > 2) return one_kernel;
    r.windows = plan_windows(N, T, kPrefillDropinScratchBytes / (int64_t(Hv) * kTileImage * 16)).count;
    if (F == 2 ? r.windows > 1 : 4 * chains * F < 3 * cus) return one_kernel;
  }
  return r;
}

// The drop-in gdn_prefill: batches of few chains with long sequences (dropin_route) on the
// two-kernel path (each chunk prepared once) in dropin_scratch; everything else, and any
// launch on a stream that is being captured into a graph, runs launch_prefill as is.
// Launches on the scratch are ordered on the device (launch_ordered), so calls on any
// streams stay correct, and calls on one stream wait for nothing they would not wait for
// anyway.
hipError_t launch_prefill_dropin(const PrefillArgs& a, hipStream_t stream) {
  const PrefillRoute r = dropin_route(a.N, a.T, a.Hv);
  if (r.windows == 0) return launch_prefill(a, stream);
  hipError_t e = hipSuccess;
  if (stream_capturing(stream, &e)) return launch_prefill(a, stream);
  if (e != hipSuccess) return e;
  return launch_ordered(a, stream, g_dropin, HIP_SYMBOL(dropin_scratch), kPrefillDropinScratchBytes, r.yields);
}

hipError_t dropin_held(hipStream_t stream, bool* held) {
  OrderedScratch* d = nullptr;
  const hipError_t e = ordered_scratch(g_dropin, &d);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> guard(d->lock);
  *held = held_by_another(*d, stream);
  return hipSuccess;
}

// gdn_prefill_no_alloc: the two-kernel path in `scratch` for batches that take it.
// On a stream that is not being captured, launches are ordered on the device like
// the drop-in's (their own event), so eager calls on any streams stay correct.  A
// launch captured into a graph cannot wait for that event: its replays and any other
// use of the array on the device must not overlap.
hipError_t launch_prefill_no_alloc(const PrefillArgs& a, hipStream_t stream) {
  const int64_t need = prefill_workspace_bytes(a.N, a.T, a.Hv);
  if (need <= 0) return launch_prefill(a, stream);
  if (need > kPrefillScratchBytes) return hipErrorInvalidValue;
  hipError_t e = hipSuccess;
  if (stream_capturing(stream, &e)) {
    PrefillArgs b = a;
    e = prefill_scratch(reinterpret_cast<void**>(&b.tiles));
    if (e != hipSuccess) return e;
    return launch_prefill(b, stream);
  }
  if (e != hipSuccess) return e;
  return launch_ordered(a, stream, g_no_alloc, HIP_SYMBOL(scratch), kPrefillScratchBytes, false);
}

// Reads (and with `reset` clears) this device's give-up count, after
// synchronising the device so that every launch so far has finished.
hipError_t prefill_giveups(uint64_t* count, bool reset) {
  hipError_t e = hipDeviceSynchronize();
  if (e != hipSuccess) return e;
  unsigned int v = 0;
  e = hipMemcpyFromSymbol(&v, HIP_SYMBOL(gdn_prefill_giveup_count), sizeof(v));
  if (e != hipSuccess) return e;
  *count = v;
  if (reset) {
    const unsigned int z = 0;
    e = hipMemcpyToSymbol(HIP_SYMBOL(gdn_prefill_giveup_count), &z, sizeof(z));
  }
  return e;
}

#ifndef GDN_PREFILL_MAX_SPLIT
#define GDN_PREFILL_MAX_SPLIT 8
#endif

namespace {
// Chains are split F ways (F a power of two, at most GDN_PREFILL_MAX_SPLIT)
// while the split grid still fits one workgroup per CU.
int split_factor(int64_t chains) {
  const int64_t cus = device_cus();
  int F = 1;
  while (F < GDN_PREFILL_MAX_SPLIT && chains * 2 * F <= cus) F *= 2;
  return F;
}

}  // namespace

int64_t prefill_work_items(int64_t chains) {
  if (chains <= 0) return 0;
  const int F = split_factor(chains);
  const int64_t grid = (chains + 15) / 16 * 16 * F;
  switch (F) {
    case 1: return grid * SplitVariant1<false>::NTHREADS;
    case 2: return grid * SplitVariant2<false>::NTHREADS;
    case 4: return grid * SplitVariant4<false>::NTHREADS;
    default: return grid * SplitVariant8<false>::NTHREADS;
  }
}

namespace {
// Largest workspace the two-kernel path uses; bigger batches take one kernel.
constexpr int64_t kMaxWorkspaceBytes = int64_t(2) << 30;
}  // namespace

// Batches split 4 or 8 ways repeat the producer work in every slice of a chain and
// are bound by it; the two-kernel path prepares each chunk once, all chunks in
// parallel, and its state pass (no producer code: 16-row consumers fit in the
// registers) runs at the consumers' pace.  Batches split 2 ways take no workspace
// (some of them gain from two kernels all the same: dropin_route), and unsplit ones
// keep producers and consumers busy on the same CUs.  The size holds the chunks of any
// offsets, also of malformed ones that overlap: N ceil(T / C) a v-head.
int64_t prefill_workspace_bytes(int N, int64_t T, int Hv) {
  if (N <= 0 || Hv <= 0 || T <= 0 || split_factor(int64_t(N) * Hv) < 4) return 0;
  const int64_t images = int64_t(N) * ((T + C - 1) / C) * Hv;
  if (images > INT32_MAX) return 0;
  const int64_t bytes = images * kTileImage * 16;
  return bytes <= kMaxWorkspaceBytes ? bytes : 0;
}

namespace {
// Launches that use the testing hooks get kernels with the hooks compiled in;
// production launches keep them out of the device code.
bool has_hooks(const PrefillArgs& a) { return a.spin_limit != 0 || a.ready_chunks != 0 || a.aborts != nullptr; }

template <bool HOOKS>
hipError_t launch_state(const PrefillArgs& a, hipStream_t stream, hipEvent_t done) {
  const int64_t chains = int64_t(a.N) * a.Hv;
  const dim3 grid(unsigned((chains + 15) / 16 * 16 * kStateSlices)), block(512);
  if (done != nullptr) {
    hipExtLaunchKernelGGL(gdn_prefill_state_kernel<HOOKS>, grid, block, 0, stream, nullptr, done, 0, a);
  } else {
    hipLaunchKernelGGL(gdn_prefill_state_kernel<HOOKS>, grid, block, 0, stream, a);
  }
  return hipGetLastError();
}

// The two-kernel path with room for `slots` chunk images a v-head (at least N), in
// plan_windows' windows, each a prep kernel and a state pass that takes the state up where
// the window before left it, in new_state: the same operations in the same order.  A window
// costs about 8 us (the launches, and both kernels filling and draining the chip); one
// 16,384-token sequence at 32 v-heads takes 412 us in two windows, 598 in one kernel.
hipError_t launch_two_kernels(const PrefillArgs& a, hipStream_t stream, int64_t slots, hipEvent_t done) {
  const int64_t tc = (a.T + C - 1) / C;
  const Windows plan = plan_windows(a.N, a.T, slots);
  const int64_t windows = plan.count, w = plan.chunks;
  // Valid offsets give at most T / C + N chunks.
  PrefillArgs b = a;
  b.prep_slots = int(tc + a.N - 1 < a.N * w ? tc + a.N - 1 : a.N * w);
  const int64_t chains = int64_t(a.N) * a.Hv;
  const bool hooks = has_hooks(a);
  for (int64_t i = 0; i < windows; ++i) {
    if (windows > 1) {
      b.win_begin = i * w * C;
      b.win_tokens = w * C;
    }
    const int64_t grid = (int64_t(b.prep_slots) * a.Hv + kPrepWaves - 1) / kPrepWaves;
    hipLaunchKernelGGL(gdn_prefill_prep_kernel, dim3(unsigned(grid)), dim3(64 * kPrepWaves), 0, stream, b);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const hipEvent_t last = i + 1 == windows ? done : nullptr;
    // (The testing hooks reach this path through a workspace, which no batch split 2 ways uses.)
    if (split_factor(chains) == 2) {
      e = launch_variant<Variant<4, 1, false, true>>(b, stream, last);
    } else if (split_factor(chains) == 4) {
      e = hooks ? launch_variant<Variant<2, 1, true, true>>(b, stream, last)
                : launch_variant<Variant<2, 1, false, true>>(b, stream, last);
    } else {
      e = hooks ? launch_state<true>(b, stream, last) : launch_state<false>(b, stream, last);
    }
    if (e != hipSuccess) return e;
    b.state = a.new_state;
  }
  return hipSuccess;
}
}  // namespace

hipError_t launch_prefill(const PrefillArgs& a, hipStream_t stream) {
  const int F = split_factor(int64_t(a.N) * a.Hv);
  if (a.tiles != nullptr && prefill_workspace_bytes(a.N, a.T, a.Hv) > 0)
    return launch_two_kernels(a, stream, a.N * ((a.T + C - 1) / C), nullptr);
  if (has_hooks(a)) {
    if (persistent_batch(a)) return launch_persistent<PersistVariant<true>>(a, stream);
    switch (F) {
      case 1: return launch_variant<SplitVariant1<true>>(a, stream);
      case 2: return launch_variant<SplitVariant2<true>>(a, stream);
      case 4: return launch_variant<SplitVariant4<true>>(a, stream);
      default: return launch_variant<SplitVariant8<true>>(a, stream);
    }
  }
  // Split chains use 16-row consumer waves (VT = 1), whose per-chunk chain is
  // shorter than a 32-row wave's.  Unsplit chains (F = 1) keep four 32-row waves:
  // eight 16-row waves and the four producers would exceed the register file.
  if (persistent_batch(a)) return launch_persistent<PersistVariant<false>>(a, stream);
  switch (F) {
    case 1: return launch_variant<SplitVariant1<false>>(a, stream);
    case 2: return launch_variant<SplitVariant2<false>>(a, stream);
    case 4: return launch_variant<SplitVariant4<false>>(a, stream);
    default: return launch_variant<SplitVariant8<false>>(a, stream);
  }
}

}  // namespace gdn

