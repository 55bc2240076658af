// Speculative verify of a Gated DeltaNet window from the read-only checkpoint
// (kernels.py:491-697 and csrc/verify.h:284-332 of the reference plugin).
//
// Per (row b, value head hv) the reference advances S <- S*d_t + c_t k_t^T
// token by token. Verify never writes the state back, so this kernel never
// forms S_t: with G_t = d_0 ... d_t,
//     S_{t-1} k_t = G_{t-1} S_0 k_t + sum_{s<t} (G_{t-1}/G_s) (k_s.k_t) c_s
//     S_t q~_t    = G_t     S_0 q~_t + sum_{s<=t} (G_t/G_s)   (k_s.q~_t) c_s
// The state enters only through the 2Q matrix-vector products
// S_0 [k_0 .. k_{Q-1}, q~_0 .. q~_{Q-1}], computed on the matrix cores
// (v_mfma_f32_4x4x1_16b_f32, FP32 in and out) from one read of the state; the
// per-row recurrence then runs on Q-vectors with the Gram matrix
// k_s.{k_t, q~_t}, evaluated incrementally (no divisions):
//     u_j <- d_t u_j + c_t (k_t.k_j),  w_j <- d_t w_j + c_t (k_t.q~_j).
//
// Work decomposition: one wave per (row, value head, TILE rows of V), TILE =
// 16, 64 or 128 (deferred commit: 16, 32 or 64) by the size of the launch
// (verify_tile in verify.hip). A
// tile is 16-row blocks streamed through two register buffers: the loads of
// blocks i+2 and i+3 are in flight while blocks i and i+1 are on the matrix
// cores, and each 64-row half runs its recurrence while the next half's loads
// are outstanding. Everything the recurrence needs from memory (v, gates) is
// loaded before the first state block, because the vector memory counter
// retires in issue order.
//
// Matrix-core layout. A 4x4x1 instruction is 16 independent blocks of a
// 4-row by 4-column outer product: lane l = 4*kb + i holds row i of A and
// column i of B of block kb, and register r of D holds (row r, column i).
// Here block kb takes the 16-byte chunks 16j + kb of four state rows (A) and of
// four of the vectors k, q~ (B) (16-bit pages of K <= 64: see RowLanes), so
//   * a load gives the 64 lanes four whole runs of 256 bytes, one per state
//     row, straight in the operand layout (the 16x16x4 instruction's layout is
//     16 rows x 64 bytes per load: half of 16 lines, which is why that form
//     needed a detour through LDS for its non-temporal loads);
//   * the B operands are the same registers for every block of rows (they
//     were re-read from LDS for each), loaded by each lane from q and k: no
//     LDS staging and no barrier before the first product;
//   * 4 columns are computed, not 16, of which Q = 4 uses 8: half the
//     matrix-core time at Q <= 4, the same at Q = 8 (see verify_wide);
//   * the Gram matrix is the same instruction on the B registers themselves.
// The 16 blocks' partial sums are added across lanes at the end of four rows
// (reduce_rows: 3 lane swaps, 3 adds and 2 rotated adds per 4x4 tile).
//
// Template parameters: S state element type, A activation type (q, k, v and
// the key record / output when they share it), KP the padded K (64, 128 or 256),
// QM window capacity (Q <= QM).
#pragma once

#include <type_traits>

#include "gdn_common.cuh"

namespace gdn {

// Element strides and page counts fit in 32 bits (checked on the host); every
// product with a row, token or page index is formed in 64 bits. The arguments
// that a wave needs before its first state load come first (see `hold` in
// verify_wave), those of the deferred commit next.
struct VerifyArgs {
  const void *qsl, *indices;
  const void *q, *k, *v, *g, *beta;
  const void *state;
  int32_t qsl_s, idx_s, qsl_i64, idx_i64;  // index dtypes: 1 for int64
  int32_t NVT, ratio;                      // tiles of a (row, value head); value heads per head
  uint32_t nvt_magic, ratio_magic;         // udiv_magic of each
  int32_t state_bs, q_ts, k_ts, v_ts, g_ts, beta_ts;
  int32_t state_hs, state_vs;
  int32_t blocks, null_block, tokens, Q, K, V;
  int32_t g_f32, beta_f32;  // 1: FP32, 0: activation dtype
  int32_t nt_rows;          // rows b < nt_rows read their state non-temporally
  // Deferred commit (kernels instantiated with DEFER): for every current row
  // the pending row it continues (p_rows), the previous step's plan arrays
  // indexed by pending row, and that step's records.
  const int32_t *p_rows, *p_src, *p_len, *p_final, *p_bnd, *p_blen;
  const float *p_corr, *p_decay;
  const void *p_key;
  int32_t p_corr_rs, p_key_rs, p_decay_rs;
  int32_t p_corr_hs, p_corr_ts, p_key_hs, p_key_ts, p_decay_hs, p_decay_ts;
  int32_t p_key_f32, p_key_per_value_head, p_record_rows, p_num_rows;
  // Read after the state loads are issued.
  float *corr;
  void *key;
  float *decay;
  void *out;
  int32_t corr_rs, key_rs, decay_rs, out_ts;
  int32_t record_rows;
  int32_t corr_hs, corr_ts, key_hs, key_ts, decay_hs, decay_ts;
  float scale;
  int32_t key_f32, out_f32;
  int32_t l2norm, key_per_value_head;
  // Fused gating: g and beta hold the raw projections a and b.
  const void *a_log, *dt_bias;
  int32_t gated, a_log_dt, dt_bias_dt;
  float softplus_beta, softplus_threshold;
};

// Division of x < 2^32 by a runtime d >= 1 with m = floor((2^32 - 1) / d): the
// high product is x / d rounded down or one less, so one correction makes it
// exact. Five scalar instructions for a uniform x; the compiler's division
// is a chain of about twenty through the vector reciprocal.
inline uint32_t udiv_magic(uint32_t d) { return 0xffffffffu / d; }
__host__ __device__ inline uint32_t udiv(uint32_t x, uint32_t d, uint32_t m) {
  const uint32_t q = uint32_t((uint64_t(x) * m) >> 32);
  return x - q * d >= d ? q + 1 : q;
}

constexpr int kVerifyThreads = 64;  // one wave per (row, value head, tile)

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <typename A>
__device__ __forceinline__ void st_f32_or(void *p, int64_t i, bool f32, float x) {
  if (f32)
    static_cast<float *>(p)[i] = x;
  else
    static_cast<A *>(p)[i] = from_f32<A>(x);
}

// Branch-free loads through buffer resources: an invalid lane passes
// kOutOfRange and reads zero, so every load of a phase issues back to back and
// no divergent branch forces a wait on it.
// Resources start at the wave's first token, so every in-bounds offset is far
// below kWindowBytes (the host checks window extents against it).
constexpr int kOutOfRange = 0x7ffff000;
constexpr int kPolicyNT = 2;  // buffer cache policy bit: non-temporal
constexpr int kWindowBytes = 0x7fff0000;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *p, int64_t byte_off) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(static_cast<const char *>(p) + byte_off), 0,
                                           kWindowBytes, 0x00020000);
}

template <typename A>
__device__ __forceinline__ float bits_to_f32(uint32_t u) {
  if constexpr (sizeof(A) == 4)
    return __uint_as_float(u);
  else
    return to_f32(__builtin_bit_cast(A, uint16_t(u)));
}

// One activation element at a byte offset (kOutOfRange reads 0).
template <typename A>
__device__ __forceinline__ float buf_ld_act(__amdgpu_buffer_rsrc_t r, int byte_off) {
  if constexpr (sizeof(A) == 4)
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, byte_off, 0, 0));
  else
    return bits_to_f32<A>(__builtin_amdgcn_raw_buffer_load_b16(r, byte_off, 0, 0));
}

// N (4 or 8) consecutive elements of a tensor that is only aligned to its
// elements. `WordRsrc` starts at the dword holding the first byte; 16-bit
// elements are read as the N/2 dwords from the one holding the first element
// and, where the run starts in a dword's upper half, one more; a funnel shift
// lines them up. Every dword read holds an element of the run.
struct WordRsrc {
  __amdgpu_buffer_rsrc_t r;
  int skip;  // bytes from the resource's start to the tensor's first byte (0 or 2)
};
__device__ __forceinline__ WordRsrc make_word_rsrc(const void *p, int64_t byte_off) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(p) + uintptr_t(byte_off);
  return {make_rsrc(reinterpret_cast<const void *>(at & ~uintptr_t(3)), 0), int(at & 2)};
}
template <typename A, int N>
struct RawRun {
  uint32_t w[sizeof(A) == 4 ? N : N / 2 + 1];
  int sh;
};
template <typename A, int N>
__device__ __forceinline__ void load_run(const WordRsrc &b, int byte_off, bool live, RawRun<A, N> &x) {
  const int off = byte_off + b.skip;
  if constexpr (sizeof(A) == 4) {
#pragma unroll
    for (int i = 0; i < N; i += 4) {
      const auto u = __builtin_amdgcn_raw_buffer_load_b128(b.r, live ? off + i * 4 : kOutOfRange, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) x.w[i + e] = u[e];
    }
  } else {
    const int at = live ? off & ~3 : kOutOfRange;
    const bool odd = (off & 2) != 0;
    if constexpr (N == 4) {
      const auto u = __builtin_amdgcn_raw_buffer_load_b64(b.r, at, 0, 0);
      x.w[0] = u[0], x.w[1] = u[1];
    } else {
      const auto u = __builtin_amdgcn_raw_buffer_load_b128(b.r, at, 0, 0);
      x.w[0] = u[0], x.w[1] = u[1], x.w[2] = u[2], x.w[3] = u[3];
    }
    x.w[N / 2] = 0u;
    // A branch of the wave: rare, and skipping it leaves fewer loads between
    // the others and the wait for them, never more.
    if (__builtin_amdgcn_ballot_w64(odd) != 0)
      x.w[N / 2] = __builtin_amdgcn_raw_buffer_load_b32(b.r, live && odd ? at + N * 2 : kOutOfRange, 0, 0);
    x.sh = odd ? 16 : 0;
  }
}
template <typename A, int N>
__device__ __forceinline__ void unpack_run(const RawRun<A, N> &x, float (&out)[N]) {
  if constexpr (sizeof(A) == 4) {
#pragma unroll
    for (int e = 0; e < N; ++e) out[e] = __uint_as_float(x.w[e]);
  } else {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      const uint32_t u = __builtin_amdgcn_alignbit(x.w[i + 1], x.w[i], x.sh);
      out[2 * i] = bits_to_f32<A>(u & 0xffffu);
      out[2 * i + 1] = bits_to_f32<A>(u >> 16);
    }
  }
}

// Wave-uniform 32-bit word through the scalar cache. Only for tensors this
// kernel never writes; the address is rounded down to a dword.
__device__ __forceinline__ uint32_t scalar_word(uintptr_t addr) {
  return *reinterpret_cast<const __attribute__((address_space(4))) uint32_t *>(addr & ~uintptr_t(3));
}

// One per-head parameter (FP32 or 16-bit) through the scalar cache.
template <typename A>
__device__ __forceinline__ float scalar_param(const void *p, int hv, int dt) {
  if (dt == GDN_DT_F32) return __uint_as_float(scalar_word(reinterpret_cast<uintptr_t>(p) + uintptr_t(hv) * 4));
  const uintptr_t addr = reinterpret_cast<uintptr_t>(p) + uintptr_t(hv) * 2;
  const uint32_t w = (scalar_word(addr) >> (int(addr & 2) * 8)) & 0xffffu;
  if (dt == GDN_DT_BF16) return __uint_as_float(w << 16);
  return float(__builtin_bit_cast(f16, uint16_t(w)));
}

template <typename S>
__device__ __forceinline__ float chunk_elem(const uint4 &raw, int e);
template <>
__device__ __forceinline__ float chunk_elem<float>(const uint4 &raw, int e) {
  return __uint_as_float(e == 0 ? raw.x : e == 1 ? raw.y : e == 2 ? raw.z : raw.w);
}
template <>
__device__ __forceinline__ float chunk_elem<bf16>(const uint4 &raw, int e) {
  const uint32_t w = (e >> 1) == 0 ? raw.x : (e >> 1) == 1 ? raw.y : (e >> 1) == 2 ? raw.z : raw.w;
  return __uint_as_float((e & 1) ? (w & 0xffff0000u) : (w << 16));
}
template <>
__device__ __forceinline__ float chunk_elem<f16>(const uint4 &raw, int e) {
  const uint32_t w = (e >> 1) == 0 ? raw.x : (e >> 1) == 1 ? raw.y : (e >> 1) == 2 ? raw.z : raw.w;
  return float(__builtin_bit_cast(f16, uint16_t((e & 1) ? (w >> 16) : (w & 0xffffu))));
}

// Orders the wave's own LDS writes before its later LDS reads. The workgroup
// is a single wave and LDS executes a wave's instructions in order, so no
// s_barrier is needed, and a wave-scope fence does not drain the outstanding
// global loads the way a workgroup barrier's release fence does.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lanes of a state row: all 16 blocks share one, except that a row of up to 64
// 16-bit elements (128 bytes) is split over 8 of them and an instruction's two
// halves take two sets of four rows. A load is then eight runs of 128 bytes, one
// line each, and a result is summed over 8 blocks; over 16 blocks half of the
// lanes and of the products were padding. K = 64, 32 heads, one layer, us over 16 /
// 8 blocks, 64-row tiles: FP16 V = 64, Q = 4, 256 rows 35.8 / 26.4; V = 192, Q = 8,
// 256 rows 163 / 105; deferred, V = 192, Q = 4, 256 rows 159 / 100.
// FP32 rows of K = 64 fill 16 blocks, and are left there: over 8 a lane holds
// twice the operands, and small launches and Q = 8 got slower (4 rows Q = 1 3.7 /
// 4.1, V = 128 256 rows Q = 8 82 / 89).
template <typename S, int KP>
struct RowLanes {
  static constexpr int E = Chunk<S>::E;       // elements per 16-byte chunk
  static constexpr int N = sizeof(S) == 2 && KP == 64 ? 8 : 16;  // blocks of a row
  static constexpr int J = KP / (N * E);      // chunks per lane per row
  static constexpr int ROWS = 64 / N;         // rows of a load
};

// The sum over a row's N blocks (16: all of kb = lane / 4, 8: kb % 8) of a value
// per (block, lane % 4), in every lane of the row.
// A rotation has no lane without a source. FOLD says so, and the move becomes part
// of the add (FP32 K = V = 128, Q = 4, 8 rows 8.6 / 8.3 us); see verify_wave for where not.
template <int CTRL, bool FOLD>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, FOLD));
}
constexpr int kRowRor8 = 0x128, kRowRor4 = 0x124;  // rotations inside 16 lanes
__device__ __forceinline__ float swap_add32(float x, float y) {  // lanes 0-31: x summed over the halves; 32-63: y
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
__device__ __forceinline__ float swap_add16(float x, float y) {  // even 16-lane rows: x summed over row pairs; odd: y
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
template <int N, bool FOLD>
__device__ __forceinline__ float sum_blocks(float x) {
  if constexpr (N == 16) x = swap_add32(x, x);
  x = swap_add16(x, x);
  return dpp_add<kRowRor4, FOLD>(dpp_add<kRowRor8, FOLD>(x));
}
// WIDE: the sum over a row's chunks c = 4j + quarter of a value per chunk, in the
// order of sum_blocks (c ^ 8, c ^ 4, c ^ 2, c ^ 1).
template <int CJ>
__device__ __forceinline__ float sum_chunks(const float (&x)[CJ]) {
  float y;
  if constexpr (CJ == 4)
    y = (x[0] + x[2]) + (x[1] + x[3]);
  else
    y = x[0] + x[1];
  y = swap_add32(y, y);
  return swap_add16(y, y);
}
// The same of CJ 16x16x1 results, register 4*(c % 4) + r: register r of the sum.
template <int CJ, typename F>
__device__ __forceinline__ f32x4 sum_results(const F &product) {  // product(j): the result of chunks 4j .. 4j + 3
  f32x16 x;
  if constexpr (CJ == 4) {
    x = product(0) + product(2);
    x += product(1) + product(3);
  } else {
    x = product(0) + product(1);
  }
  f32x4 y;
#pragma unroll
  for (int r = 0; r < 4; ++r) y[r] = (x[r] + x[8 + r]) + (x[4 + r] + x[12 + r]);
  return y;
}
// The sum for the four registers of a 4x4 result tile at once. N = 16: lane
// 16*r + 4*any + i gets the sum of row r, column i. N = 8: `lo` gets rows 0 (lanes
// of even 16) and 1 (odd), `hi` rows 2 and 3, each half of the wave its own tile.
template <bool FOLD>
__device__ __forceinline__ float reduce_rows(f32x4 a) {
  const float x = swap_add16(swap_add32(a[0], a[2]), swap_add32(a[1], a[3]));
  return dpp_add<kRowRor4, FOLD>(dpp_add<kRowRor8, FOLD>(x));
}
template <bool FOLD>
__device__ __forceinline__ void reduce_rows8(f32x4 a, float &lo, float &hi) {
  lo = dpp_add<kRowRor4, FOLD>(dpp_add<kRowRor8, FOLD>(swap_add16(a[0], a[1])));
  hi = dpp_add<kRowRor4, FOLD>(dpp_add<kRowRor8, FOLD>(swap_add16(a[2], a[3])));
}

// DEFER: before verifying, apply the previous step's commit for this row (the
// fold of kernels.py:1222-1324, folded into the next verify): the state comes
// from the pending commit's source page, its accepted prefix is replayed from
// the previous step's records block by block, the result is stored to the
// final page (and the boundary snapshot to the boundary page), and the window
// is verified from the folded values, rounded to the state type exactly as
// the stored page is. Each state page is read once per step instead of twice.
// The wave's LDS, declared once per kernel and shared by both cache-policy
// bodies below (a __shared__ array inside each would be allocated twice).
template <int QM, int KP, bool DEFER, int TILE, int STAGE>
struct __align__(16) VerifyLds {
  static constexpr int HALF = TILE < 64 ? TILE : 64;
  uint4 stage[STAGE];         // one block of rows on its way to the 16x16x1 layout
  float d[HALF][2 * QM + 1];  // GEMV results of one half tile
  __align__(16) float pk[DEFER ? QM : 1][DEFER ? KP : 1];  // pending commit's keys
  float pc[DEFER ? QM : 1][DEFER ? HALF : 1];              // and its corrections of the tile's rows
};

// Rows of a block: 16, or 8 where the two block buffers (128 registers a lane at
// 16 rows) and the 64 registers of B operands of FP32 pages of K > 128 at Q > 4
// would take a wave all its SIMD's registers: at 16 rows that kernel had one
// wave per SIMD, or spilled (K = 256, Q = 8, 32 heads, 64 rows: 143 us held to
// three waves, 69 to two, 65 with blocks of 8 rows).
template <typename S, int KP>
__host__ __device__ constexpr int verify_block_rows(int qm) {
  return sizeof(S) == 4 && KP == 256 && qm == 8 ? 8 : 16;
}

// Windows of more than four tokens have 16 columns: a 16x16x1 instruction of four
// blocks (one per quarter of the wave) takes the same matrix-core time as 4x4x1
// ones, and its partial sums meet in a lane's own registers, 60 adds per 16 rows
// instead of 160 cross-lane instructions. Tiles of 64 rows and up whose rows are at
// most 256 bytes are bound by instructions there, so their blocks go through LDS
// into that layout (lane l holds row l % 16, chunks 4j + l / 16): one write and one
// read per load of 1 KiB. Products and sums keep the 4x4x1 form's order, so that a
// row's result does not depend on the launch it is in. One layer of 32 heads, Q = 8,
// us with 4x4x1 / 16x16x1: FP16 K = V = 128, 64 rows 34.4 / 29.5, 256 rows 108 / 91; FP16
// K = 64, V = 192, 256 rows 103 / 85; BF16 K = 64, V = 128, 256 rows 68 / 61; FP32 K = 64,
// V = 128, 32 rows 18.8 / 15.4, 256 rows 81 / 75. Tiles of 16 rows are a chain of latencies
// that the detour lengthens (BF16 K = 128, 4 rows 7.4 / 9.0), and the deferred verify is
// bound by its fold (BF16 K = 128, 64 rows 54.6 / 58.0).
template <typename S, int KP>
__host__ __device__ constexpr bool verify_wide(int qm, bool defer, int tile) {
  return qm == 8 && !defer && tile >= 64 && KP * int(sizeof(S)) <= 256;
}
template <typename S, int KP>
__host__ __device__ constexpr int verify_stage(int qm, bool defer, int tile) {  // chunks of a staged block
  return verify_wide<S, KP>(qm, defer, tile) ? 16 * KP / Chunk<S>::E : 1;
}

template <typename S, typename A, int KP, int QM, bool DEFER, bool NT, int TILE>
__device__ __forceinline__ void verify_wave(const VerifyArgs &a,
                                            VerifyLds<QM, KP, DEFER, TILE, verify_stage<S, KP>(QM, DEFER, TILE)> &L) {
  static_assert(!DEFER || TILE <= 64, "the pending corrections cover one half tile");
  using R = RowLanes<S, KP>;
  constexpr int E = R::E, J = R::J;    // elements of a chunk, chunks per lane per row
  constexpr int NV = 2 * QM;           // columns: k_0 .. k_{QM-1}, q~_0 .. q~_{QM-1}
  constexpr bool WIDE = verify_wide<S, KP>(QM, DEFER, TILE);
  constexpr int CW = WIDE ? 16 : 4;            // columns of a group: one instruction's
  constexpr int CG = (NV + CW - 1) / CW;       // groups of columns
  constexpr int CGK = (QM + CW - 1) / CW;      // column groups that hold a k
  constexpr int CN = WIDE ? 4 : R::N;          // lanes that share a column's vector
  constexpr int CJ = KP / (CN * E);            // chunks of it per lane
  // Rotated adds as one instruction, but in the kernel whose scalars the compiler
  // then spills around every block (K = 256, 32 heads, 1 row 6.2 us, folded 6.7).
  constexpr bool FOLD = !(sizeof(S) == 4 && KP == 256 && QM == 4 && TILE == 16 && !DEFER);
  constexpr bool MIXED = QM % CW != 0;         // a group may hold k and q columns
  constexpr int BROWS = verify_block_rows<S, KP>(QM);
  constexpr int BG = BROWS / R::ROWS;  // loads of a block per chunk
  constexpr int NRB = TILE / BROWS;    // blocks per tile
  constexpr int HALF = TILE < 64 ? TILE : 64;  // rows of one recurrence (one per lane)
  constexpr int HRB = HALF / BROWS;
  auto &d_lds = L.d;
  auto &pk_lds = L.pk;
  auto &pc_lds = L.pc;

  // One batch of argument reads: left to itself the compiler reads each
  // argument where it is first used, one wait per read, ahead of the state
  // loads. The asm is one consumer of them all.
  asm volatile("" ::"s"(a.qsl), "s"(a.indices), "s"(a.q), "s"(a.k), "s"(a.v), "s"(a.g), "s"(a.beta), "s"(a.state),
               "s"(a.qsl_s), "s"(a.idx_s), "s"(a.qsl_i64), "s"(a.idx_i64), "s"(a.NVT), "s"(a.ratio), "s"(a.nvt_magic),
               "s"(a.ratio_magic), "s"(a.state_bs), "s"(a.q_ts), "s"(a.k_ts), "s"(a.v_ts), "s"(a.g_ts),
               "s"(a.beta_ts), "s"(a.state_hs), "s"(a.state_vs), "s"(a.blocks), "s"(a.null_block), "s"(a.tokens),
               "s"(a.Q), "s"(a.K), "s"(a.V));
  const int hv = int(udiv(blockIdx.x, uint32_t(a.NVT), a.nvt_magic));
  const int vt = int(blockIdx.x) - hv * a.NVT;
  const int b = int(blockIdx.y);
  const int ratio = a.ratio;
  const int h = int(udiv(uint32_t(hv), uint32_t(ratio), a.ratio_magic));
  const int lane = threadIdx.x;
  const int V = a.V, K = a.K;
  const int row0 = vt * TILE;
  const int Q = a.Q;
  constexpr int AS = int(sizeof(A));

  // ---- 0. the wave's metadata: one lane-indexed load, one wait ----
  // Lanes 0-5: low and high words of query_start_loc[b], query_start_loc[b+1]
  // and state_indices[b]; DEFER: lane 6 the pending row of b.
  int64_t bos, eos, slot;
  int prow = 0;
  {
    const uintptr_t q0 = elem_addr(a.qsl, int64_t(b) * a.qsl_s, a.qsl_i64);
    const uintptr_t q1 = elem_addr(a.qsl, int64_t(b + 1) * a.qsl_s, a.qsl_i64);
    const uintptr_t s0 = elem_addr(a.indices, int64_t(b) * a.idx_s, a.idx_i64);
    const uintptr_t hq = a.qsl_i64 ? 4 : 0, hs = a.idx_i64 ? 4 : 0;
    uintptr_t addr = q0;
    addr = lane == 1 ? q0 + hq : addr;
    addr = lane == 2 ? q1 : addr;
    addr = lane == 3 ? q1 + hq : addr;
    addr = lane == 4 ? s0 : addr;
    addr = lane == 5 ? s0 + hs : addr;
    if constexpr (DEFER) addr = lane == 6 ? reinterpret_cast<uintptr_t>(a.p_rows) + uintptr_t(b) * 4u : addr;
    const uint32_t w = lane_word(addr);
    bos = index_of(word_of(w, 0), word_of(w, 1), a.qsl_i64);
    eos = index_of(word_of(w, 2), word_of(w, 3), a.qsl_i64);
    slot = index_of(word_of(w, 4), word_of(w, 5), a.idx_i64);
    if constexpr (DEFER) prow = int(word_of(w, 6));
  }
  const int64_t qlen = eos - bos;
  const int64_t out_base = int64_t(hv) * V + row0;
  // Token validity is uniform across the wave (kernels.py:612): lane t < QM
  // tests token t and one ballot gathers the window's mask (an unrolled test
  // per token became a chain of scalar branches).
  uint32_t valid_mask;
  {
    const int64_t tok = bos + lane;
    const bool tv = lane < QM && lane < Q && lane < qlen && tok >= 0 && tok < a.tokens;
    valid_mask = uint32_t(__builtin_amdgcn_ballot_w64(tv));
  }

  // ---- 1. gates (and DEFER: the pending plan and decays): one load ----
  // Lane t < QM reads the dword holding g of token t, lane QM + t that of
  // beta (FP32, or the 16-bit value at its half); every address is formed on
  // its own lane. Tokens outside the window read the first word of
  // query_start_loc (always present; g and beta may be empty, hence null,
  // when the launch has no token at all) and are discarded. DEFER: lanes
  // 2QM .. 2QM+4 read the pending row's accepted length, source, final and
  // boundary pages and boundary length, and lanes 2QM+5 .. 3QM+4 its decays;
  // a row without a pending row reads row 0 (num_rows >= 1) and discards it.
  // The ordinary kernel waits for these words only after its state loads
  // issue; the deferred one needs the pending source page first.
  const int gsz = a.g_f32 ? 4 : AS, bsz = a.beta_f32 ? 4 : AS;
  const uintptr_t any_word = reinterpret_cast<uintptr_t>(a.qsl);
  const bool gate_lane_b = lane >= QM;          // lanes QM .. 2QM-1 carry beta
  const int gate_t = (gate_lane_b ? lane - QM : lane) & 31;
  int gate_sh;                                   // bit offset of this lane's 16-bit gate in its word
  uint32_t gw;
  const bool prow_ok = DEFER && prow >= 0 && prow < a.p_num_rows && prow < a.p_record_rows;
  const int pr = prow_ok ? prow : 0;
  {
    const bool tv = lane < 2 * QM && ((valid_mask >> gate_t) & 1u);
    const uintptr_t base = reinterpret_cast<uintptr_t>(gate_lane_b ? a.beta : a.g);
    const int64_t ts = gate_lane_b ? a.beta_ts : a.g_ts;
    const int64_t sz = gate_lane_b ? bsz : gsz;
    uintptr_t addr = tv ? base + uintptr_t(((bos + gate_t) * ts + hv) * sz) : any_word;
    gate_sh = int(addr & 2) * 8;
    if constexpr (DEFER) {
      const int32_t *plan[5] = {a.p_len, a.p_src, a.p_final, a.p_bnd, a.p_blen};
#pragma unroll
      for (int i = 0; i < 5; ++i)
        addr = lane == 2 * QM + i ? reinterpret_cast<uintptr_t>(plan[i] + pr) : addr;
      const int dt = lane - (2 * QM + 5);
      const uintptr_t da = reinterpret_cast<uintptr_t>(a.p_decay) +
                           uintptr_t((int64_t(pr) * a.p_decay_rs + int64_t(hv) * a.p_decay_hs +
                                      int64_t(dt) * a.p_decay_ts) * 4);
      addr = dt >= 0 && dt < QM ? (dt < Q ? da : any_word) : addr;
    }
    // A relaxed atomic load is an ordinary one that the compiler leaves here: it
    // moved the plain load down to its use, behind the state loads, and waiting
    // for it was then waiting for all of them.
    gw = __hip_atomic_load(reinterpret_cast<const __attribute__((address_space(1))) uint32_t *>(addr & ~uintptr_t(3)),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  }

  // Pending commit of the previous step (same validity rule as the fold,
  // kernels.py:1232-1242 / csrc/fold.h:192-205). The row continues pending
  // row `prow` (plan and record row of the previous step) only when its state
  // index names that commit's final page: a row whose request is new, or
  // whose metadata names another page, verifies from its own page and leaves
  // the pending commit to a flush.
  bool pend = false, pstore_b = false;
  int pn = 0, pblen = 0;
  int64_t psrc = 0, pfin = 0, pbnd = 0;
  if constexpr (DEFER) {
    pn = int(word_of(gw, 2 * QM + 0));
    psrc = int(word_of(gw, 2 * QM + 1));
    pfin = int(word_of(gw, 2 * QM + 2));
    pbnd = int(word_of(gw, 2 * QM + 3));
    pblen = int(word_of(gw, 2 * QM + 4));
    pend = prow_ok && pn > 0 && pn <= Q && psrc > a.null_block && psrc < a.blocks && pfin > a.null_block &&
           pfin < a.blocks && pfin == slot;
    pstore_b = pend && pbnd > a.null_block && pbnd < a.blocks && pbnd != pfin && pblen > 0 && pblen <= pn;
    prow = pend ? prow : 0;  // record addressing below stays inside the records
  }
  const int pend_len = pend ? pn : 0;  // tokens of the pending commit to replay
  const bool null_slot = slot <= a.null_block || slot >= a.blocks;
  if (null_slot) {
    // Null or out-of-range page: zero outputs for the window, records untouched
    // (kernels.py:569-583).
    for (int t = 0; t < Q; ++t) {
      const int64_t tok = bos + t;
      if (!(t < qlen && tok >= 0 && tok < a.tokens)) continue;
      for (int r = lane; r < TILE; r += kVerifyThreads)
        if (row0 + r < V) st_f32_or<A>(a.out, tok * a.out_ts + out_base + r, a.out_f32 != 0, 0.0f);
    }
    return;  // a pending commit needs slot == its final page, never a null one
  }
  if (valid_mask == 0 && !pend) return;
  // A pending commit on a row with nothing to verify still has to be applied:
  // that wave runs the whole pipeline with no token (every input load reads
  // out of range and nothing but the folded tile is stored).
  const bool verify_row = !null_slot && valid_mask != 0;
  if (!verify_row) valid_mask = 0;

  // Block within its row, row / column within its 4, and the row's place in a load.
  const int kb = (lane >> 2) & (R::N - 1), ij = lane & 3, lr = R::N == 16 ? ij : 4 * (lane >> 5) + ij;
  const int bq = (lane >> 2) & 3;  // a result's copy (reduce_rows)
  const int cl = WIDE ? lane & 15 : ij, cs = WIDE ? lane >> 4 : kb;  // column in its group, first chunk of its vector

  // ---- 2. small loads first: the lane's chunks of k and q, v of its rows ----
  // Column c = CW*cg + cl is k_c, or q_{c - QM}.
  const WordRsrc rq = make_word_rsrc(a.q, bos * a.q_ts * AS), rk = make_word_rsrc(a.k, bos * a.k_ts * AS);
  RawRun<A, E> raw_q[CG][CJ], raw_k[CG][CJ];
#pragma unroll
  for (int cg = 0; cg < CG; ++cg) {
    const int col = CW * cg + cl;
    const bool is_q = col >= QM;
    const int t = (is_q ? col - QM : col) & 31;
    // Non-short-circuit tests: a short-circuit chain became a branch per load,
    // with kernel arguments reloaded inside it.
    const bool on = (col < NV) & (((valid_mask >> t) & 1u) != 0);
#pragma unroll
    for (int j = 0; j < CJ; ++j) {
      const int kk = (CN * j + cs) * E;
      const int off = (t * (is_q ? a.q_ts : a.k_ts) + h * K + kk) * AS;
      // A group is all k or all q, or one of two loads reads out of range.
      if (MIXED || CW * cg < QM) load_run<A, E>(rk, off, on & !is_q & (kk < K), raw_k[cg][j]);
      if (MIXED || CW * cg >= QM) load_run<A, E>(rq, off, on & is_q & (kk < K), raw_q[cg][j]);
    }
  }
  // DEFER: the pending commit's keys (token t, 4 elements from kk) for LDS, FP32
  // or activation-typed records (one of the two loads reads out of range),
  // and its corrections of the lane's row.
  constexpr int C4 = KP / 4;
  constexpr int PK_PASSES = DEFER ? (QM * C4 + kVerifyThreads - 1) / kVerifyThreads : 1;
  RawRun<float, 4> pk32[PK_PASSES];
  RawRun<A, 4> pka[PK_PASSES];
  float pcx[QM];
  if constexpr (DEFER) {
    const int key_head = a.p_key_per_value_head ? hv : h;
    const int64_t kbase = int64_t(prow) * a.p_key_rs + int64_t(key_head) * a.p_key_hs;
    const bool kf32 = a.p_key_f32 != 0;
    const WordRsrc rpk = make_word_rsrc(a.p_key, kbase * (kf32 ? 4 : AS));
    int lim = pend_len;
    asm volatile("" : "+v"(lim));  // per-lane select, not a branch
#pragma unroll
    for (int p = 0; p < PK_PASSES; ++p) {
      const int idx = p * kVerifyThreads + lane;
      const int t = idx / C4, kk = (idx - t * C4) * 4;
      const bool live = (t < lim) & (kk < K);
      const int el = t * a.p_key_ts + kk;
      load_run<float, 4>(rpk, el * 4, live & kf32, pk32[p]);
      load_run<A, 4>(rpk, el * AS, live & !kf32, pka[p]);
    }
    const __amdgpu_buffer_rsrc_t rpc =
        make_rsrc(a.p_corr, (int64_t(prow) * a.p_corr_rs + int64_t(hv) * a.p_corr_hs + row0) * 4);
    const int row_lim = ((lane < HALF) & (row0 + lane < V)) ? lim : 0;
#pragma unroll
    for (int t = 0; t < QM; ++t)
      pcx[t] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
          rpc, t < row_lim ? (t * a.p_corr_ts + lane) * 4 : kOutOfRange, 0, 0));
  }
  // v of the lane's row in each half; the second half is loaded later, after
  // the loads it must not wait behind.
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(a.v, bos * a.v_ts * AS);
  float vv[2][QM];
  auto load_v = [&](int half) {
#pragma unroll
    for (int t = 0; t < QM; ++t) {
      const int vr = row0 + half * 64 + lane;
      const bool ok = (vr < V) & (lane < HALF) & (((valid_mask >> t) & 1u) != 0);
      const int off = ok ? (t * int(a.v_ts) + int(out_base) + half * 64 + lane) * AS : kOutOfRange;
      vv[half][t] = buf_ld_act<A>(rv, off);
    }
  };
  load_v(0);

  // ---- 3. first two state blocks ----
  // Buffer loads: one resource per (slot, head) tile, a 32-bit per-lane offset
  // per chunk and the block step in the scalar offset. Rows >= V lie past the
  // resource's extent and read as zero; chunks >= K get an out-of-range offset.
  // Register g*J + j of a block: row ROWS*g + lr, chunk N*j + kb.
  const int tile_rows = V - row0 < TILE ? V - row0 : TILE;
  const int tile_bytes = tile_rows * a.state_vs * int(sizeof(S));
  auto tile_rsrc = [&](int64_t page, bool use) {
    const S *tp = static_cast<const S *>(a.state) + page * a.state_bs + int64_t(hv) * a.state_hs +
                  int64_t(row0) * a.state_vs;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<S *>(use ? tp : static_cast<const S *>(a.state)), 0,
                                             use ? tile_bytes : 0, 0x00020000);
  };
  // DEFER with a pending commit: read the pending source page; the folded
  // tile goes to the final page (and its snapshot to the boundary page).
  const __amdgpu_buffer_rsrc_t rsrc = tile_rsrc(pend ? psrc : slot, true);
  const __amdgpu_buffer_rsrc_t rfin = tile_rsrc(pfin, pend);
  const __amdgpu_buffer_rsrc_t rbnd = tile_rsrc(pbnd, pstore_b);
  const int row_bytes = a.state_vs * int(sizeof(S));
  // A 24-bit product (row_bytes < 2^24, checked on the host): a full multiply
  // here became a 64-bit multiply-add whose unused high addend was a register
  // with a load in flight, and waiting for it held back the first state loads.
  const int lane_off = int(__umul24(unsigned(lr), unsigned(row_bytes))) + kb * 16;
  constexpr int BR = BG * J;  // 16-byte chunks per lane of a block
  auto s_voff = [&](int j) { return (R::N * j + kb) * E < K ? lane_off : kOutOfRange; };
  auto s_soff = [&](int rb, int g, int j) { return (rb * BROWS + R::ROWS * g) * row_bytes + j * R::N * 16; };
  // One form for every K, and every block is loaded (blocks past V read as
  // zero): a conditional load would leave a path on which it was not issued,
  // and the wait counts of every later MFMA would have to assume that path,
  // draining the pipeline at each block.
  auto load_block = [&](int rb, uint4 (&dst)[BR]) {
#pragma unroll
    for (int g = 0; g < BG; ++g)
#pragma unroll
      for (int j = 0; j < J; ++j)
        dst[g * J + j] = __builtin_bit_cast(
            uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, s_voff(j), s_soff(rb, g, j), NT ? kPolicyNT : 0));
  };
  uint4 bufA[BR], bufB[BR];
  __builtin_amdgcn_sched_barrier(0);  // the gates' load (and every other small one) stays ahead of the state
  load_block(0, bufA);
  __builtin_amdgcn_sched_barrier(0);  // keep block 0's loads ahead of block 1's
  if constexpr (NRB > 1) load_block(1, bufB);
  // The rest, with the arguments it needs behind `z`.
  auto rest = [&](const auto *z) __attribute__((always_inline)) {
  float dec[QM], bet[QM];
  float neg_a = 0.0f, dtb = 0.0f;
  if (z->gated) {
    neg_a = -expf(scalar_param<A>(z->a_log, hv, z->a_log_dt));
    dtb = scalar_param<A>(z->dt_bias, hv, z->dt_bias_dt);
  }
  {
    // Each gate lane decodes its own word; the window's decays and betas then
    // reach every lane by readlane.
    const bool f32 = gate_lane_b ? z->beta_f32 != 0 : z->g_f32 != 0;
    float x = f32 ? __uint_as_float(gw) : bits_to_f32<A>((gw >> gate_sh) & 0xffffu);
    if (z->gated) {
      // docs/reference/recoverssm_gdn_upstream.py:135-151
      if (gate_lane_b) {
        x = 1.0f / (1.0f + expf(-x));
      } else {
        const float xb = x + dtb;
        const float bx = z->softplus_beta * xb;
        const float sp = bx <= z->softplus_threshold ? log1pf(expf(bx)) / z->softplus_beta : xb;
        x = neg_a * sp;
      }
    }
    const float gate = gate_lane_b ? x : expf(x);
#pragma unroll
    for (int t = 0; t < QM; ++t) {
      const bool tv = (valid_mask >> t) & 1u;
      dec[t] = tv ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gate), t)) : 1.0f;
      bet[t] = tv ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gate), QM + t)) : 0.0f;
    }
  }

  // ---- 4. operands, records, Gram matrix ----
  const bool rec_ok = b < z->record_rows;
  const bool key_writer = rec_ok && vt == 0 && (z->key_per_value_head || hv == h * ratio);
  float m[CG][CJ][E];  // the lane's chunks of its columns' vectors (B operands)
#pragma unroll
  for (int cg = 0; cg < CG; ++cg)
#pragma unroll
    for (int j = 0; j < CJ; ++j) {
      if constexpr (MIXED) {
        // One of the two was read out of range, as zeros. Their words are ORed:
        // a sum would lose the sign of a zero, and the key record holds the
        // key's own bits.
        RawRun<A, E> x = raw_k[cg][j];
#pragma unroll
        for (int i = 0; i < int(sizeof(x.w) / 4); ++i) x.w[i] |= raw_q[cg][j].w[i];
        if constexpr (sizeof(A) == 2) x.sh = CW * cg + cl >= QM ? raw_q[cg][j].sh : x.sh;
        unpack_run<A, E>(x, m[cg][j]);
      } else {
        unpack_run<A, E>(CW * cg < QM ? raw_k[cg][j] : raw_q[cg][j], m[cg][j]);
      }
    }
  if (z->l2norm) {
    // kernels.py:645-648: x * rsqrt(sum(x*x) + 1e-6) for q and k, then q *= scale.
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
      float ss[CJ] = {};  // WIDE: of each chunk
#pragma unroll
      for (int j = 0; j < CJ; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) ss[WIDE ? j : 0] = __builtin_fmaf(m[cg][j][e], m[cg][j][e], ss[WIDE ? j : 0]);
      float total;
      if constexpr (WIDE)
        total = sum_chunks(ss);
      else
        total = sum_blocks<R::N, FOLD>(ss[0]);
      const float inv = rsqrtf(total + 1e-6f);
#pragma unroll
      for (int j = 0; j < CJ; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) m[cg][j][e] *= inv;
    }
  }
  if (key_writer) {
    const int key_head = z->key_per_value_head ? hv : h;
    const bool key_f32 = z->key_f32 != 0;
#pragma unroll
    for (int cg = 0; cg < CGK; ++cg) {
      const int t = CW * cg + cl;
      if (t < QM && ((valid_mask >> (t & 31)) & 1u) && (WIDE || R::N == 16 || lane < 32)) {  // N = 8: both halves hold it
#pragma unroll
        for (int j = 0; j < CJ; ++j) {
          const int kk = (CN * j + cs) * E;
          if (kk < K) {
            const int64_t base = int64_t(b) * z->key_rs + int64_t(key_head) * z->key_hs + int64_t(t) * z->key_ts + kk;
#pragma unroll
            for (int e = 0; e < E; ++e) st_f32_or<A>(z->key, base + e, key_f32, m[cg][j][e]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int cg = QM / CW; cg < CG; ++cg) {
    const float sc = CW * cg + cl >= QM ? z->scale : 1.0f;
#pragma unroll
    for (int j = 0; j < CJ; ++j)
#pragma unroll
      for (int e = 0; e < E; ++e) m[cg][j][e] *= sc;
  }
  if (rec_ok && vt == 0) {
    float dl = 1.0f;
#pragma unroll
    for (int t = 0; t < QM; ++t) dl = lane == t ? dec[t] : dl;
    if (lane < QM && ((valid_mask >> lane) & 1u))
      z->decay[int64_t(b) * z->decay_rs + int64_t(hv) * z->decay_hs + int64_t(lane) * z->decay_ts] = dl;
  }
  // k_s . column c in lane gram_lane(s, c) of gram[s / 4][c / 4]; WIDE: of
  // wide_gram[s % 4] (lane l, register r: row 4*(l / 16) + r, column l % 16).
  auto gram_lane = [](int s, int c) {
    return WIDE ? 16 * (s >> 2) + c : (R::N == 16 ? 16 * (s & 3) : 16 * (s & 1) + 4 * ((s >> 1) & 1)) + (c & 3);
  };
  float gram[WIDE ? 1 : CGK][WIDE ? 1 : CG];
  f32x4 wide_gram = {0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (WIDE) {
    wide_gram = sum_results<CJ>([&](int j) {
      f32x16 acc = {};
#pragma unroll
      for (int e = 0; e < E; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x1f32(m[0][j][e], m[0][j][e], acc, 0, 0, 0);
      return acc;
    });
  } else {
#pragma unroll
    for (int s = 0; s < CGK; ++s)
#pragma unroll
      for (int cg = 0; cg < CG; ++cg) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int e = 0; e < E; ++e) acc = __builtin_amdgcn_mfma_f32_4x4x1f32(m[s][j][e], m[cg][j][e], acc, 0, 0, 0);
        if constexpr (R::N == 16) {
          gram[s][cg] = reduce_rows<FOLD>(acc);
        } else {
          float lo, hi;
          reduce_rows8<FOLD>(acc, lo, hi);
          gram[s][cg] = (bq & 1) != 0 ? hi : lo;
        }
      }
  }
  auto dot = [&](int s, int c) {
    const float x = WIDE ? wide_gram[s & 3] : gram[WIDE ? 0 : s / 4][WIDE ? 0 : c / 4];
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), gram_lane(s, c)));
  };
  // DEFER: the pending keys and corrections to LDS, the decays to scalars. A
  // lane's chunks of the keys stay in registers where they are few.
  constexpr bool PK_REGS = DEFER && QM * J * E <= 32;
  float pdec[QM];
  float pkr[PK_REGS ? QM : 1][PK_REGS ? J : 1][E];
  if constexpr (DEFER) {
#pragma unroll
    for (int p = 0; p < PK_PASSES; ++p) {
      const int idx = p * kVerifyThreads + lane;
      const int t = idx / C4, kk = (idx - t * C4) * 4;
      float x32[4], xa[4];
      unpack_run<float, 4>(pk32[p], x32);
      unpack_run<A, 4>(pka[p], xa);
      if (t < QM) {
#pragma unroll
        for (int e = 0; e < 4; ++e) pk_lds[t][kk + e] = x32[e] + xa[e];
      }
    }
#pragma unroll
    for (int t = 0; t < QM; ++t) {
      if (lane < HALF) pc_lds[t][lane] = pcx[t];
      const bool live = pend && t < pn;
      pdec[t] = live ? __uint_as_float(word_of(gw, 2 * QM + 5 + t)) : 1.0f;
    }
    wave_lds_sync();
    if constexpr (PK_REGS) {
#pragma unroll
      for (int t = 0; t < QM; ++t)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int e = 0; e < E; ++e) pkr[t][j][e] = pk_lds[t][(R::N * j + kb) * E + e];
    }
  }

  // DEFER: replay the pending accepted prefix on one block in registers,
  // h <- fma(c_t, k_t, h * d_t) as the fold does, storing the boundary snapshot
  // after `boundary_len` tokens and the final state after n (kernels.py:1242-1324).
  // The final store is issued on every path (an unused one falls out of
  // range) so the wait counts of the loads in flight do not depend on the row;
  // the boundary snapshot's only on rows that have one (about one tile in
  // seven at B=256).
  auto fold_block = [&](int rb, uint4 (&buf)[BR]) {
    if constexpr (DEFER) {
      const int seg = pstore_b ? pblen : 0;
      // FP32 values of the lane's chunks; the fold keeps them in FP32 across
      // the boundary snapshot and rounds only what it stores, as the fold does.
      float h[BR][E];
#pragma unroll
      for (int i = 0; i < BR; ++i) unpack16<S>(buf[i], h[i]);
      auto apply = [&](int lo, int hi) {
#pragma unroll
        for (int t = 0; t < QM; ++t) {
          if (t >= lo && t < hi) {
            const float d = pdec[t];
            float c[BG];
#pragma unroll
            for (int g = 0; g < BG; ++g) c[g] = pc_lds[t][(rb & (HRB - 1)) * BROWS + R::ROWS * g + lr];
#pragma unroll
            for (int j = 0; j < J; ++j) {
              float kv[E];
#pragma unroll
              for (int e = 0; e < E; ++e) {
                if constexpr (PK_REGS)
                  kv[e] = pkr[t][j][e];
                else
                  kv[e] = pk_lds[t][(R::N * j + kb) * E + e];
              }
#pragma unroll
              for (int g = 0; g < BG; ++g)
#pragma unroll
                for (int e = 0; e < E; ++e) h[g * J + j][e] = __builtin_fmaf(c[g], kv[e], h[g * J + j][e] * d);
            }
          }
        }
      };
      auto store = [&](__amdgpu_buffer_rsrc_t r) {
        // Non-temporal row runs, as loaded (see the deferred rule in verify.hip).
#pragma unroll
        for (int g = 0; g < BG; ++g)
#pragma unroll
          for (int j = 0; j < J; ++j)
            store_b128_settled<NT ? kPolicyNT : 0>(__builtin_bit_cast(gdn_u32x4, pack16<S>(h[g * J + j])), r,
                                                   s_voff(j), s_soff(rb, g, j));
      };
      apply(0, seg);
      if (pstore_b) store(rbnd);
      apply(seg, pn);
      store(rfin);
      // The window is verified from the folded tile as stored.
#pragma unroll
      for (int i = 0; i < BR; ++i) buf[i] = pack16<S>(h[i]);
    }
  };

  // ---- 5. pipelined S_0 . [k, q~] on the matrix cores, recurrence per half ----
  // WIDE: a block's chunk c of row r sits at r*CPR + (c ^ swz(r)) of the stage: 16
  // consecutive lanes of a write, and the 16 rows a read takes of one chunk, are
  // in 16 different places modulo 256 bytes.
  constexpr int CPR = KP / E;
  auto stage_slot = [](int row, int c) {
    return row * CPR + (c ^ (CPR == 16 ? ((row & 3) << 2) | (row >> 2) : ((row & 2) << 1) | (row >> 2)));
  };
  auto stage_block = [&](const uint4 (&src)[BR]) {
    static_assert(!WIDE || (BROWS == 16 && J == 1 && (CPR == 16 || CPR == 8)), "stage_slot's rows");
    wave_lds_sync();  // the block before has been read
#pragma unroll
    for (int g = 0; g < BG; ++g) L.stage[stage_slot(R::ROWS * g + lr, kb)] = src[g];
    wave_lds_sync();
  };
  auto wide_block = [&](int rb) {
    uint4 op[CJ];
#pragma unroll
    for (int j = 0; j < CJ; ++j) op[j] = L.stage[stage_slot(cl, 4 * j + cs)];
    const f32x4 acc = sum_results<CJ>([&](int j) {
      f32x16 x = {};
#pragma unroll
      for (int e = 0; e < E; ++e)
        x = __builtin_amdgcn_mfma_f32_16x16x1f32(chunk_elem<S>(op[j], e), m[0][j][e], x, 0, 0, 0);
      return x;
    });
    const int row = (rb & (HRB - 1)) * BROWS + 4 * cs;
#pragma unroll
    for (int i = 0; i < 4; ++i) d_lds[row + i][cl] = acc[i];
  };
  auto gemv_block = [&](int rb, const uint4 (&src)[BR]) {
    float y[CG];
#pragma unroll
    for (int g = 0; g < BG; ++g) {
      f32x4 acc[CG];
#pragma unroll
      for (int cg = 0; cg < CG; ++cg) acc[cg] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float x = chunk_elem<S>(src[g * J + j], e);
#pragma unroll
          for (int cg = 0; cg < CG; ++cg)
            acc[cg] = __builtin_amdgcn_mfma_f32_4x4x1f32(x, m[cg][j][e], acc[cg], 0, 0, 0);
        }
      // Every copy holds the sums; one keeps them: copy g those of rows 4g .. 4g+3
      // (N = 16), copies 2g and 2g + 1 those of rows 8g + {0, 1} and 8g + {2, 3} of
      // each half's four.
#pragma unroll
      for (int cg = 0; cg < CG; ++cg) {
        if constexpr (R::N == 16) {
          const float r = reduce_rows<FOLD>(acc[cg]);
          y[cg] = g == 0 || bq == g ? r : y[cg];
        } else {
          float lo, hi;
          reduce_rows8<FOLD>(acc[cg], lo, hi);
          y[cg] = g == 0 || bq == 2 * g ? lo : y[cg];
          y[cg] = bq == 2 * g + 1 ? hi : y[cg];
        }
      }
    }
    const int row = (rb & (HRB - 1)) * BROWS +
                    (R::N == 16 ? 4 * bq + (lane >> 4)
                                : 8 * (bq >> 1) + 4 * (lane >> 5) + 2 * (bq & 1) + ((lane >> 4) & 1));
#pragma unroll
    for (int cg = 0; cg < CG; ++cg)
      if ((BROWS == 16 || bq < BG) && (NV % 4 == 0 || 4 * cg + ij < NV)) d_lds[row][4 * cg + ij] = y[cg];
  };
  // Outputs and corrections go out through buffer stores that are issued for
  // every token and lane (an invalid one gets an out-of-range offset and is
  // dropped): a store skipped on some path would make the wait counts of the
  // loads still in flight assume it, and drain the pipeline at the next block.
  const bool out_f32 = z->out_f32 != 0;
  const __amdgpu_buffer_rsrc_t rout = make_rsrc(z->out, (bos * z->out_ts + out_base) * (out_f32 ? 4 : AS));
  const __amdgpu_buffer_rsrc_t rcorr =
      make_rsrc(z->corr, (int64_t(b) * z->corr_rs + int64_t(hv) * z->corr_hs + row0) * 4);
  float res_c[2][QM], res_o[2][QM];  // corrections and outputs of the lane's row in each half
  auto emit = [&](int half) {
    const int lrow = half * 64 + lane;
    int row_ok = (row0 + lrow < V) & (lane < HALF);
    asm volatile("" : "+v"(row_ok));  // per-lane offsets below, not branches
#pragma unroll
    for (int t = 0; t < QM; ++t) {
      const bool st = ((valid_mask >> t) & 1u) && row_ok;
      const int oel = t * int(z->out_ts) + lrow;
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(res_o[half][t]), rout,
                                            st && out_f32 ? oel * 4 : kOutOfRange, 0, 0);
      if constexpr (sizeof(A) == 2)
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, from_f32<A>(res_o[half][t])), rout,
                                              st && !out_f32 ? oel * AS : kOutOfRange, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(res_c[half][t]), rcorr,
                                            st && rec_ok ? (t * z->corr_ts + lrow) * 4 : kOutOfRange, 0, 0);
    }
  };
  auto recurrence = [&](int half) {
    wave_lds_sync();  // d_lds complete
    float u[QM], wq[QM];
#pragma unroll
    for (int t = 0; t < QM; ++t) {
      u[t] = d_lds[lane & (HALF - 1)][t];
      wq[t] = d_lds[lane & (HALF - 1)][QM + t];
    }
#pragma unroll
    for (int t = 0; t < QM; ++t) {
      const bool tv = (valid_mask >> t) & 1u;
      const float d = dec[t];
      const float c = tv ? (vv[half][t] - d * u[t]) * bet[t] : 0.0f;
      if (tv) {
#pragma unroll
        for (int j = t + 1; j < QM; ++j) u[j] = __builtin_fmaf(c, dot(t, j), d * u[j]);
#pragma unroll
        for (int j = t; j < QM; ++j) wq[j] = __builtin_fmaf(c, dot(t, QM + j), d * wq[j]);
      }
      res_c[half][t] = c;
      res_o[half][t] = wq[t];
    }
    emit(half);
    wave_lds_sync();  // d_lds may be overwritten by the next half
  };
#pragma unroll
  for (int rb = 0; rb < NRB; rb += 2) {
    // A staged block's registers are free before its products.
    fold_block(rb, bufA);
    if constexpr (WIDE)
      stage_block(bufA);
    else
      gemv_block(rb, bufA);
    if (rb + 2 < NRB) load_block(rb + 2, bufA);
    if constexpr (WIDE) wide_block(rb);
    if constexpr (NRB > 1) {
      fold_block(rb + 1, bufB);
      if constexpr (WIDE)
        stage_block(bufB);
      else
        gemv_block(rb + 1, bufB);
      if (rb + 3 < NRB) load_block(rb + 3, bufB);
      if constexpr (WIDE) wide_block(rb + 1);
    }
    if (TILE == 128 && rb + 2 == NRB / 2) load_v(1);  // smaller tiles have no second half
    // Every half runs its recurrence, also one past V (its rows store nothing):
    // skipping it would be a path without its stores.
    constexpr int PASS = HRB < 2 ? 2 : HRB;  // blocks of a half, taken two at a time
    if ((rb + 2) % PASS == 0) recurrence((rb + 2) / PASS - 1);
  }
  };
  if constexpr (TILE == 128) {
    // Long tiles: the rest's arguments are read where they are used, not with
    // the others at the kernel's start, from where they were held in spilled
    // registers (12 layers of 64 rows: verify + commit 909 against 922 us).
    // Short tiles are a chain of latencies, and the reads lengthened it (24
    // layers of 16 rows: 534 against 512 us).
    const auto *z = (const __attribute__((address_space(4))) VerifyArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(z));
    rest(z);
  } else {
    rest(&a);
  }
}

// Rows b < a.nt_rows read their state tiles with non-temporal loads, the
// rest with ordinary ones. A launch streams its tiles once; what an ordinary
// load leaves in the memory-side cache is what a commit reading the same pages
// right after finds there, and only the last-read part of a large batch can
// still be there. Reading the earlier part non-temporally keeps it from
// evicting that part (and the non-temporal reads run faster): the host sets
// nt_rows so that the ordinary reads cover the last `retain` bytes.
// Long tiles keep three waves per SIMD (168 registers) where they fit: left
// free, Q = 8 at K = 128 takes 184 registers and two waves (B=256 step 306
// against 287 us); four waves spill (318 us). They fit where the two block
// buffers and the B operands take at most 96 registers; past that (FP32 pages of
// K > 128, 16-bit ones at Q > 4) three waves spilled, and the bound is two (K =
// 256, 32 heads of V = 128, us with three waves / two: FP32 pages Q = 4, 128 rows
// 152 / 103, Q = 1 99 / 90; BF16 pages Q = 8, 128 rows 100 / 94). So it is where FP32
// activations meet the 16x16x1 form's accumulators on rows of 128 16-bit elements.
// Shorter tiles ask for two waves, which leaves a wave 256 registers and none of
// the accumulation file: with one, products were copied out of it (Q = 8: FP32 K =
// 64, V = 192, 256 rows 122 / 113 us; K = V = 128, deferred, 64 rows 71 / 68; Q = 4:
// FP32 K = 256, 8 rows 12.7 / 12.0; FP16 K = 96, V = 192, 29 rows of 12 heads 11.0 /
// 10.4). Not those it made slower, the ordinary BF16 tile of K = 128 at Q = 4 (32 rows
// 14.6 / 15.1), nor 16 rows at Q <= 4 (no difference) and K > 128 at Q <= 2, where the
// compiler spilled more scalars for it, nor the deferred FP16 kernels of K > 128 at
// Q > 4, which do not fit.
template <typename S, typename A, int KP>
constexpr int verify_min_waves(int qm, int tile, bool defer) {
  using R = RowLanes<S, KP>;
  const int buffers = 2 * (verify_block_rows<S, KP>(qm) / R::ROWS) * R::J * 4;
  const int operands = (2 * qm + 3) / 4 * R::J * R::E;
  const bool wide_f32 = verify_wide<S, KP>(qm, defer, tile) && KP == 128 && sizeof(A) == 4;
  if (tile == 128) return buffers + operands <= 96 && !wide_f32 ? 3 : 2;
  if (qm == 8) return defer && KP == 256 && std::is_same_v<S, f16> ? 1 : 2;
  if (tile == 16 || (KP == 256 && qm <= 2)) return 1;
  return !defer && KP == 128 && qm == 4 && std::is_same_v<S, bf16> ? 1 : 2;
}
template <typename S, typename A, int KP, int QM, bool DEFER, int TILE>
__global__ __launch_bounds__(kVerifyThreads, (verify_min_waves<S, A, KP>(QM, TILE, DEFER))) void verify_kernel(
    VerifyArgs a) {
  __shared__ VerifyLds<QM, KP, DEFER, TILE, verify_stage<S, KP>(QM, DEFER, TILE)> lds;
  warm_kernel_args<int(sizeof(VerifyArgs))>();
  if (DEFER || int(blockIdx.y) < a.nt_rows)  // the deferred verify: every row (see verify.hip)
    verify_wave<S, A, KP, QM, DEFER, true, TILE>(a, lds);
  else
    verify_wave<S, A, KP, QM, DEFER, false, TILE>(a, lds);
}

// Launch for one state type; defined per state type in verify_<state>.hip.
template <typename S>
void launch_verify_state(int act_dt, int kp, int tile, int qm, bool deferred, dim3 grid, hipStream_t s,
                         const VerifyArgs &a);

template <typename S, typename A, int KP, bool DEFER, int TILE>
static void launch_verify_q(int qm, dim3 grid, hipStream_t s, const VerifyArgs &a) {
  const dim3 wg(kVerifyThreads);
  switch (qm) {
    case 1: hipLaunchKernelGGL((verify_kernel<S, A, KP, 1, DEFER, TILE>), grid, wg, 0, s, a); break;
    case 2: hipLaunchKernelGGL((verify_kernel<S, A, KP, 2, DEFER, TILE>), grid, wg, 0, s, a); break;
    case 4: hipLaunchKernelGGL((verify_kernel<S, A, KP, 4, DEFER, TILE>), grid, wg, 0, s, a); break;
    default: hipLaunchKernelGGL((verify_kernel<S, A, KP, 8, DEFER, TILE>), grid, wg, 0, s, a); break;
  }
}

template <typename S, typename A, int KP, bool DEFER>
static void launch_verify_tile(int tile, int qm, dim3 grid, hipStream_t s, const VerifyArgs &a) {
  switch (tile) {
    case 16: launch_verify_q<S, A, KP, DEFER, 16>(qm, grid, s, a); break;
    case 64: launch_verify_q<S, A, KP, DEFER, 64>(qm, grid, s, a); break;
    default: launch_verify_q<S, A, KP, DEFER, DEFER ? 32 : 128>(qm, grid, s, a); break;
  }
}

template <typename S, typename A, bool DEFER>
static void launch_verify_kp(int kp, int tile, int qm, dim3 grid, hipStream_t s, const VerifyArgs &a) {
  switch (kp) {
    case 64: launch_verify_tile<S, A, 64, DEFER>(tile, qm, grid, s, a); break;
    case 128: launch_verify_tile<S, A, 128, DEFER>(tile, qm, grid, s, a); break;
    default: launch_verify_tile<S, A, 256, DEFER>(tile, qm, grid, s, a); break;
  }
}

template <typename S, bool DEFER>
static void launch_verify_act(int act_dt, int kp, int tile, int qm, dim3 grid, hipStream_t s, const VerifyArgs &a) {
  switch (act_dt) {
    case GDN_DT_BF16: launch_verify_kp<S, bf16, DEFER>(kp, tile, qm, grid, s, a); break;
    case GDN_DT_F16: launch_verify_kp<S, f16, DEFER>(kp, tile, qm, grid, s, a); break;
    default: launch_verify_kp<S, float, DEFER>(kp, tile, qm, grid, s, a); break;
  }
}

// The deferred-commit kernels of each state type live in a translation unit of
// their own (verify_<state>_deferred.hip), so the halves compile in parallel.
template <typename S>
void launch_verify_deferred(int act_dt, int kp, int tile, int qm, dim3 grid, hipStream_t s, const VerifyArgs &a);

#define GDN_DEFINE_VERIFY_LAUNCH(STATE)                                                                \
  template <>                                                                                          \
  void launch_verify_state<STATE>(int act_dt, int kp, int tile, int qm, bool deferred, dim3 grid, hipStream_t s, \
                                  const VerifyArgs &a) {                                               \
    if (deferred)                                                                                      \
      launch_verify_deferred<STATE>(act_dt, kp, tile, qm, grid, s, a);                                        \
    else                                                                                               \
      launch_verify_act<STATE, false>(act_dt, kp, tile, qm, grid, s, a);                                      \
  }

#define GDN_DEFINE_VERIFY_DEFERRED_LAUNCH(STATE)                                                         \
  template <>                                                                                            \
  void launch_verify_deferred<STATE>(int act_dt, int kp, int tile, int qm, dim3 grid, hipStream_t s,                \
                                     const VerifyArgs &a) {                                              \
    launch_verify_act<STATE, true>(act_dt, kp, tile, qm, grid, s, a);                                           \
  }

}  // namespace gdn
