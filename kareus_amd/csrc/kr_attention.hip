// Causal grouped-query flash attention for head dimensions 128 and 64 on the gfx950 matrix cores.
//
// Roofline: MFMA.  Algorithmic work: forward 2*b*nq*s^2*hd FLOP (causal half of 4*s^2*hd),
// backward 2.5x that.
//
// Forward (attn_fwd_pp_kernel below).  A workgroup of 8 waves owns 128 consecutive queries of
// one (batch, query head); wave w and wave w + 4 own the same 32 of them and walk the even /
// odd 64-key tiles, in antiphase, merging their softmax partials at the end.
//   S^T = K . Q^T is computed with K rows on the MFMA A port and the wave's Q fragment (held
//   in registers for the whole kernel) on the B port, so a lane ends up with 16 scores per
//   32-key tile *of a single query row* (row = lane % 32; lanes l and l+32 split the keys).
//   The online-softmax row maximum and row sum are therefore in-lane reductions plus one
//   exchange between the two half-waves.
//   O^T += V^T . P^T: the probabilities are already laid out as the B-port operand (the
//   contraction index of an MFMA can be permuted freely as long as both operands agree), and
//   V^T fragments come out of LDS through the transposing read ds_read_b64_tr_b16.  Neither
//   P nor V is ever transposed through memory.
// Tensors are addressed through (seq, batch, head) strides, so sequence-major [s, b, h, d]
// views of the fused QKV projection are consumed in place.
#include <initializer_list>

#include "kr_common.h"

namespace {

constexpr int HD = 128;
constexpr int BQ = 128;       // queries per workgroup (4 waves x 32, twice over)
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
// Online softmax of the MFMA forward kernels: a row's exponents are taken against a reference
// point that follows the running maximum only when the maximum has grown by more than this many
// powers of two.  In between, probabilities run up to 2^8 instead of 1 — rounding is relative in
// fp32 and in bf16, the row sum and the output carry the same factor and the final division takes
// it out — and the 64 accumulator multiplies of a rescale are skipped (with 32 rows per wave some
// row's maximum moves in most tiles; by more than 2^8 it hardly ever does after the first).
constexpr float kRescaleSlack = 8.0f;
constexpr int kXcds = 8;

// Workgroup -> (rank of its tile by the length of its causal rows or columns, 0 the longest; (batch, head) pair).  An XCD has a
// contiguous range of the pairs' tiles, so that what pairs share stays in its L2, and starts with the longest of all its pairs:
// short ones fill up the units that finish first.  With more than sixteen pairs (and more than two workgroups for each of its 32
// units) what the pairs read no longer fits the L2: 32 / ntiles of them start at once, and the others follow.
// Rows of each pair in sequence -> this order, us, dQ, forward and dK/dV at head dimension 128: 3 x 2008 tokens of 8/2 heads 67
// -> 54, 58 -> 45, 92 -> 84; dK/dV 6 x 4096 of 3/1 heads 249 -> 180, 4 x 4096 of 24/8 heads 867 -> 843; two pairs at once -> this
// order, 2 x 8192 of 32/8 heads forward 1016 -> 978, dQ 1363 -> 1330.  All pairs at once beyond sixteen: 64 x 512 tokens of 32/8
// heads forward 276 -> 300, dK/dV 366 -> 411.  Where every workgroup has a unit to itself all start at once, and where pairs are
// one tile there is nothing to order; the divisions only delay them: one pair after the other (256 tokens of 8/8 heads of 64 forward
// 9.6 -> 9.3, dQ 8.0 -> 7.7; 512 tokens of 8/2 heads 11.9 -> 11.6, 10.5 -> 10.3).
// The choice is the launch's: the first order permutes the ids of one XCD, the second those of groups that cross from one XCD's
// range into the next, so that only all of them together take every tile once.  (The XCDs' shares differ by one workgroup.)
__device__ __forceinline__ void longest_first(int pid, int nblocks, int ntiles, int& rank, int& pair) {
  const int q = nblocks / kXcds, r = nblocks % kXcds, xcd = pid % kXcds;
  const int first = xcd * q + (xcd < r ? xcd : r), count = q + (xcd < r ? 1 : 0), i = pid / kXcds;
  const int most = q + (r > 0 ? 1 : 0);  // workgroups of the XCD with the most
  if (most <= 32 || ntiles == 1) {  // a unit for every workgroup, or tiles of one length
    rank = (first + i) % ntiles;
    pair = (first + i) / ntiles;
    return;
  }
  if (most <= 64 || most <= 16 * ntiles) {
    // ids first .. first + count - 1, id = pair * ntiles + rank: every rank `full` times, `extra` ranks from that of the
    // first id on (cyclically) once more.  Ranks [0, a) occur na times, [a, b) nb times, the others na times again.
    const int start = first % ntiles, full = count / ntiles, extra = count - full * ntiles;
    const bool wraps = start + extra > ntiles;
    const int a = wraps ? start + extra - ntiles : start, b = wraps ? start : start + extra;
    const int na = wraps ? full + 1 : full, nb = wraps ? full : full + 1;
    int at = i, from = 0, n = na;
    if (at >= a * na) {
      at -= a * na;
      from = a;
      n = nb;
      if (at >= (b - a) * nb) {
        at -= (b - a) * nb;
        from = b;
        n = na;
      }
    }
    const int row = at / n;
    rank = from + row;
    const int ahead = rank - start;
    pair = (first + (ahead < 0 ? ahead + ntiles : ahead)) / ntiles + (at - row * n);
    return;
  }
  const int lid = first + i, total_pairs = nblocks / ntiles;
  const int grp = (ntiles < 32 && 32 % ntiles == 0) ? 32 / ntiles : 1;
  const int span = grp * ntiles, base = lid / span, at = lid % span;
  if ((base + 1) * grp <= total_pairs) {
    rank = at / grp;
    pair = base * grp + at % grp;
  } else {  // a last, incomplete group keeps the plain order
    rank = lid % ntiles;
    pair = lid / ntiles;
  }
}

// Output staging.  After the MFMAs a lane holds, for its row (lane % 32), groups of four
// consecutive channels; stored from there an instruction scatters 64 small pieces over 32 rows
// and the texture-address path takes them one at a time.  Each wave therefore passes its
// results through 4 KB of LDS of its own (32 rows of 128 bytes, 16-byte chunks XOR-swizzled
// against bank conflicts) and reads them back as whole rows, 8 lanes per row, so an
// instruction writes 8 contiguous 128-byte segments.  Only lanes of one wave exchange data:
// the program order of its LDS instructions is all the ordering needed.
struct RowStage {
  char* base;
  int wr, wsw, h, rrow, rch;
  __device__ __forceinline__ void init(void* lds4k, int lane) {
    base = reinterpret_cast<char*>(lds4k);
    const int r = lane & 31;
    h = lane >> 5;
    wr = r * 128;
    wsw = (r >> 1) & 7;
    rrow = lane >> 3;
    rch = lane & 7;
  }
  static __device__ __forceinline__ void sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  }
  // bf16 pass = 32 rows x 64 channels: block j (0/1) of 32 channels, group g of the MFMA layout
  __device__ __forceinline__ void put_bf16(int j, int g, bf16x4 v) const {
    *reinterpret_cast<bf16x4*>(base + wr + (((4 * j + g) ^ wsw) << 4) + 8 * h) = v;
  }
  // read q (0..3): row 8q + lane/8 of the pass, channels 8*(lane%8) .. +7
  __device__ __forceinline__ bf16x8 get_bf16(int q, int& row, int& col) const {
    row = 8 * q + rrow;
    col = 8 * rch;
    return *reinterpret_cast<const bf16x8*>(base + row * 128 + ((rch ^ ((row >> 1) & 7)) << 4));
  }
  // fp32 pass = 32 rows x 32 channels
  __device__ __forceinline__ void put_f32(int g, f32x4 v) const {
    *reinterpret_cast<f32x4*>(base + wr + (((2 * g + h) ^ wsw) << 4)) = v;
  }
  __device__ __forceinline__ f32x4 get_f32(int q, int& row, int& col) const {
    row = 8 * q + rrow;
    col = 4 * rch;
    return *reinterpret_cast<const f32x4*>(base + row * 128 + ((rch ^ ((row >> 1) & 7)) << 4));
  }
};

// 32 rows x D channels of fp32 accumulators (scaled) -> bf16 rows at dst + row * row_stride; RAGGED: only the
// first `valid` rows exist
template <int D, bool RAGGED>
__device__ __forceinline__ void store_rows_bf16(const RowStage& st, const f32x16 (&acc)[D / 32],
                                                float mul, bf16* dst, int64_t row_stride, int valid) {
#pragma unroll
  for (int pass = 0; pass < D / 64; ++pass) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (bf16)(acc[2 * pass + j][g * 4 + e] * mul);
        st.put_bf16(j, g, v);
      }
    RowStage::sync();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int row, col;
      const bf16x8 v = st.get_bf16(q, row, col);
      if (!RAGGED || row < valid) stg8(dst + (int64_t)row * row_stride + pass * 64 + col, v);
    }
    RowStage::sync();
  }
}

// the same as fp32 rows (partial results for a later reduction)
template <int D>
__device__ __forceinline__ void store_rows_f32(const RowStage& st, const f32x16 (&acc)[D / 32],
                                               float mul, float* dst, int64_t row_stride) {
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[dt][g * 4 + e] * mul;
      st.put_f32(g, v);
    }
    RowStage::sync();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int row, col;
      const f32x4 v = st.get_f32(q, row, col);
      *reinterpret_cast<f32x4*>(dst + (int64_t)row * row_stride + dt * 32 + col) = v;
    }
    RowStage::sync();
  }
}

}  // namespace

static int check_attn_common(int s, int b, int nq, int nkv, int hd) {
  if (s <= 0 || b <= 0 || nq <= 0 || nkv <= 0) return KR_EINVAL;
  if (hd <= 0 || hd % 8 || hd > 128 || nq % nkv) return KR_EUNSUPPORTED;
  if (b > 65535 || nq > 65535) return KR_EUNSUPPORTED;  // grid dimensions of the general kernels
  return KR_OK;
}
// The training workloads' shapes: head dimension 128 and whole 128-row tiles.
static bool attn_fast_path(int s, int hd) { return hd == HD && s % BQ == 0; }
// The MFMA kernels also take head dimension 64 and ragged lengths as they lie (template parameters D and
// RAGGED), provided that a lane's byte offset to any row of a 128-row tile fits 32 bits.  The alternative is to
// copy into padded buffers of 128 channels and whole tiles and back (nine to eleven small launches, and half
// of the matrix work on zeros where D = 64).  Measured, padded -> in place, forward / backward in us:
//   s 256, b 1, 8/8 heads of 64       28 / 57     ->   9 / 22     (launches)
//   s 2048, b 1, 32/8 heads of 64     75 / 190    ->  35 / 100
//   s 4096, b 2, 32/8 heads of 64    282 / 909    -> 171 / 495    (0.80 / 0.69 PFLOP/s)
//   s 776, b 1, 8/2 heads of 128      31 / 78     ->  20 / 53
//   s 4000, b 4, 8/2 heads of 128    167 / 532    -> 145 / 485    (whole tiles, s 4096: 133 / 470)
//   s 8184, b 2, 32/8 heads of 128  1121 / 3744   -> 1092 / 3623
// Other head dimensions, and strides beyond that bound, are still padded.
static bool attn_in_place(int s, int hd, std::initializer_list<int64_t> seq_strides) {
  if (attn_fast_path(s, hd)) return true;
  if (hd != 128 && hd != 64) return false;
  for (int64_t ss : seq_strides)
    if (127 * ss + 128 >= ((int64_t)1 << 31)) return false;
  return true;
}

static int kr_compute_units() {
  static const int num_cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    return n;
  }();
  return num_cus;
}

// The kernels keep a sequence stride in 32 bits and build per-lane byte offsets of up to
// (48 * stride + 128) * 2 from it: strides must be positive and small enough for that.
template <size_t N>
inline bool attn_strides_ok(const int64_t (&seq)[N], std::initializer_list<int64_t> others) {
  for (int64_t ss : seq)
    if (ss <= 0 || 48 * ss + 128 >= ((int64_t)1 << 31)) return false;
  for (int64_t st : others)
    if (st <= 0) return false;
  return true;
}

// =============================================================================================
// Backward.  Launches: delta pre-pass, dK/dV pass, (group reduction), dQ pass — or, with 256-query
// tiles, the one-wave dQ kernel first (it computes delta itself), then dK/dV and the group
// reduction.  No atomics, deterministic.
//   1. delta[b, h, i] = sum_d dO[i, d] * O[i, d]                      (HBM-bound pre-pass; kept negated)
//   2. dK, dV: a workgroup owns 128 keys of one (batch, QUERY head) — 32 per pair of waves,
//      their K and V fragments in the registers of the pair's score wave, dK and dV in those of
//      its accumulate wave — and streams every query tile at or below the diagonal through LDS.
//      Per 32x32 block:
//        S = Q.K^T, dP = dO.V^T (rows = queries on the MFMA A port, so a lane holds one key
//        column), P = exp2(S*c - lse), dS = P*(dP - delta), then dV^T += dO^T.P and
//        dK^T += Q^T.dS with the Q / dO tiles read back transposed (ds_read_b64_tr_b16).
//      With grouped-query attention several query heads share a KV head: each workgroup
//      writes an fp32 partial for its query head and a small HBM-bound kernel sums the
//      partials of a group (one query head per KV head: bf16 results are written directly).
//      Splitting by query head rather than looping over the group keeps enough workgroups in
//      flight when one GPU holds only a few KV heads (a tensor-parallel shard).
//   3. dQ: a workgroup owns 128 queries of one (batch, head) and streams the key tiles up to
//      the diagonal: S^T = K.Q^T, dP^T = V.dO^T (a lane holds one query row), dS^T, then
//      dQ^T += K^T.dS^T with the K tile read back transposed.
//   Recomputing S and dP in both passes costs 7 instead of 5 tile products but keeps every
//   accumulator in registers and every output written exactly once.
// Every K / V / Q / dO tile is staged straight from global memory into a blocked LDS tile that
// can be read both ways (as rows and transposed) without bank conflicts; see bt_request below.
// =============================================================================================
namespace {


// query-like tensors: head h of KV group g = h / per sits at g*g_ + (h % per)*h_
struct QLayout {
  int64_t s_, b_, g_, h_;
  __device__ __forceinline__ int64_t at(int bi, int head, int per) const {
    return (int64_t)bi * b_ + (head / per) * g_ + (head % per) * h_;
  }
};
struct KLayout {
  int64_t s_, b_, h_;
  __device__ __forceinline__ int64_t at(int bi, int kvh) const { return (int64_t)bi * b_ + kvh * h_; }
};

// Scalar loads return out of order, so while one is pending (a kernel argument fetched in the
// prologue and first used behind the loop is, as far as the compiler's wait-count pass knows, for
// the whole loop) every wait for an LDS read becomes lgkmcnt(0): the first MFMA of a group then
// waits for the fragments of the next group too.  An explicit lgkmcnt(0) in front of a loop ends
// that: inside, the waits count.
__device__ __forceinline__ void settle_scalar_loads() { __builtin_amdgcn_s_waitcnt(0xc07f); }

// ---- direct global -> LDS loads (see the GEMM for why they are written as inline assembly:
// the compiler must not know of them, or it drains them in front of every barrier).  The 64
// lanes of one load land contiguously: lane p at lds_byte + 16 p.
__device__ __forceinline__ void dma_b128(const void* base, uint32_t byte_off, uint32_t lds_byte) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_byte), "v"(byte_off), "s"(base)
               : "memory", "m0");
}

// 4 bytes per lane: lane p lands at lds_byte + 4 p
__device__ __forceinline__ void dma_b32(const void* base, uint32_t byte_off, uint32_t lds_byte) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :
               : "s"(lds_byte), "v"(byte_off), "s"(base)
               : "memory", "m0");
}

// ---- blocked LDS tile: [64 rows][128 channels] bf16, filled straight from global memory ------
// A tile is 16 blocks; block B holds rows r, r+16, r+32, r+48 (r = 4 (B % 4) + B / 4), 256 bytes
// each, in the order one wave-wide request delivers them (lane p at +16 p: row r + 16 (p / 16),
// 16-byte chunk p % 16 — 16 consecutive lanes fetch one contiguous row), then 16 bytes of
// padding.  Both ways of reading fragments out of it are free of bank conflicts, and every
// fragment address is one per-lane base plus an instruction immediate.
constexpr uint32_t BT_BLK = 1024 + 16, BT_BYTES = 16 * BT_BLK;

// Head dimension 64: the same image holds 128 rows of 64 channels.  Image row i is row i of the tile
// followed by row i + 64 (chunks 0-7 and 8-15), so requests, bank behaviour and the number of MFMAs a
// tile feeds are those of 64 rows of 128 channels, and only the lane's source address and the fragment
// immediates differ: 32-row block t of the tile sits in image rows 32 (t % 2) .., column half t / 2.
// (Figures against padding the heads to 128 channels: at attn_in_place.)
template <int D>
constexpr int tile_rows = 64 * 128 / D;

// row of the tile (relative to the request's first row) and channel a lane fetches
template <int D>
__device__ __forceinline__ int tile_lane_row(int lane) {
  return (lane >> 4) * 16 + (D == 64 ? ((lane >> 3) & 1) * 64 : 0);
}
template <int D>
__device__ __forceinline__ int tile_lane_ch(int lane) {
  return (lane & (D / 8 - 1)) * 8;
}
template <int D>
__device__ __forceinline__ uint32_t tile_lane_off(int lane, int ss) {
  return (uint32_t)(tile_lane_row<D>(lane) * ss + tile_lane_ch<D>(lane)) * 2u;
}

// A tile that reaches beyond the sequence (rows row0 .. of `origin`, s rows exist): every lane's row is
// clamped into the sequence for the request, and once it has landed the wave overwrites the rows
// beyond s with zeros (zero_tail), before the barrier that publishes the tile.  `r` is the request's first
// row within the tile.  Only the last tiles of a ragged sequence take this road.
template <int D>
__device__ __forceinline__ void request_clamped(const bf16* origin, int64_t ss, int row0, int r, int s, int lane,
                                                uint32_t lds) {
  const int base = row0 < s - 1 ? row0 : s - 1;
  const int key = r + tile_lane_row<D>(lane), last = s - 1 - base;
  dma_b128(origin + (int64_t)base * ss,
           (uint32_t)((key < last ? key : last) * (int)ss + tile_lane_ch<D>(lane)) * 2u, lds);
}
template <int D>
__device__ __forceinline__ void zero_block_tail(int row0, int r, int s, int lane, uint32_t lds) {
  if (row0 + r + tile_lane_row<D>(lane) >= s) *(KR_LDS bf16x8*)(lds + lane * 16) = zero8();
}

// The four waves (wave = 0..3) of a group bring in one tile; `rows` = its first row in global
// memory.  Wave w fills blocks w, w + 4, w + 8, w + 12, which hold the tile rows 4 w + 0..3
// (+ 16, 32, 48): four consecutive rows, so a request costs one pointer increment.
template <int D>
__device__ __forceinline__ void bt_request(const bf16* rows, int64_t ss, uint32_t tile, int wave,
                                           int lane) {
  int l2 = lane;
  asm volatile("" : "+v"(l2));  // nothing derived from it is kept alive between requests
  const uint32_t lane_off = tile_lane_off<D>(l2, (int)ss);
  const bf16* row = rows + (int64_t)(4 * wave) * ss;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    dma_b128(row, lane_off, tile + (wave + 4 * i) * BT_BLK);
    row += ss;
  }
}
// the same for a tile that may reach beyond the sequence, and the zeros behind its rows (see request_clamped)
template <int D>
__device__ __forceinline__ void bt_request_clamped(const bf16* origin, int64_t ss, int row0, int s, uint32_t tile,
                                                   int wave, int lane) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    request_clamped<D>(origin, ss, row0, 4 * wave + i, s, lane, tile + (wave + 4 * i) * BT_BLK);
}
template <int D>
__device__ __forceinline__ void bt_zero_tail(int row0, int s, uint32_t tile, int wave, int lane) {
#pragma unroll
  for (int i = 0; i < 4; ++i) zero_block_tail<D>(row0, 4 * wave + i, s, lane, tile + (wave + 4 * i) * BT_BLK);
}
// row-major fragments: lane gets row 32 t + lane % 32, channels 16 kk + 8 (lane / 32) + 0..7
__device__ __forceinline__ uint32_t bt_rows_lane(int lane) {
  const int r = lane & 31;
  return (uint32_t)((4 * (r & 3) + ((r >> 2) & 3)) * BT_BLK + (r >> 4) * 256 + (lane >> 5) * 16);
}
template <int D>
__device__ __forceinline__ bf16x8 bt_rows(uint32_t base, int t, int kk) {
  return *(KR_LDS const bf16x8*)(base + (t & 1) * 512 + (t >> 1) * 128 + kk * 32);
}
// transposed fragments: lane gets channel 32 dt + lane % 32, rows 16 g + {4 h + 0..3, 8 + 4 h + 0..3}
__device__ __forceinline__ uint32_t bt_cols_lane(int lane) {
  const int p = lane & 15;
  return (uint32_t)((4 * (p >> 2) + (lane >> 5)) * BT_BLK + ((lane >> 4) & 1) * 32 +
                    ((p & 3) >> 1) * 16 + (p & 1) * 8);
}
template <int D>
__device__ __forceinline__ bf16x8 bt_cols(uint32_t base, int g, int dt) {
  union {
    struct { s16x4 lo, hi; } s;
    bf16x8 v;
  } u;
  const uint32_t a = base + (g & 3) * 256 + (g >> 2) * 128 + dt * 64;
  u.s.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((KR_LDS s16x4*)(a));
  u.s.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((KR_LDS s16x4*)(a + 2 * BT_BLK));
  return u.v;
}

// Ping-pong forward.  Two halves of four waves own the same 128 queries and walk the even / odd
// key tiles (their partial softmax results are merged at the end, half 1 handing its state to
// half 0 through LDS), but the halves run in antiphase.  Time is cut into periods by workgroup
// barriers; in every period one half only feeds the matrix pipe — P.V of its previous tile, then
// S = Q.K^T of its next one, 32 MFMAs — while the other half does everything else for its own
// tile: the softmax (exponentials, row statistics, rounding to bf16, the occasional rescale of
// the output accumulators) and the requests for the K / V tiles two steps ahead, which go
// straight from global memory into blocked [64][128] LDS tiles.  A SIMD hosts one wave of each
// half, so its matrix pipe and its vector ALU are busy at the same time instead of taking
// turns, which is what happens when co-resident waves are in the same phase.
template <int D, bool RAGGED>
__global__ __launch_bounds__(512, 1) void attn_fwd_pp_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    bf16* __restrict__ o, float* __restrict__ lse, int s, int nq, int nkv, float scale_log2,
    int64_t q_ss, int64_t q_sb, int64_t q_sg, int64_t q_sh, int64_t k_ss, int64_t k_sb,
    int64_t k_sh, int64_t v_ss, int64_t v_sb, int64_t v_sh, int64_t o_ss, int64_t o_sb,
    int64_t o_sg, int64_t o_sh) {
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];
  constexpr int NB = tile_rows<D> / 32;  // 32-key blocks of a tile
  constexpr int DT = D / 32, KK = D / 16;
  constexpr int TK = tile_rows<D>;       // keys of a tile

  const int half = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
  const int tid = threadIdx.x & 255;
  const int lane = tid & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nqt = (s + BQ - 1) / BQ;
  int rank, pair;
  longest_first(blockIdx.x, gridDim.x, nqt, rank, pair);
  const int qt = nqt - 1 - rank;
  const int head = pair % nq;
  const int bi = pair / nq;
  const int per = nq / nkv;
  const int kvh = head / per, hj = head % per;

  const int q0 = qt * BQ;
  const int qw0 = q0 + wave * 32;
  const int qrow = qw0 + (lane & 31);
  const bf16* qp = q + (int64_t)bi * q_sb + kvh * q_sg + hj * q_sh +
                   (int64_t)(RAGGED && qrow >= s ? s - 1 : qrow) * q_ss;
  const bf16* kb = k + (int64_t)bi * k_sb + (int64_t)kvh * k_sh;
  const bf16* vb = v + (int64_t)bi * v_sb + (int64_t)kvh * v_sh;

  bf16x8 qf[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) qf[kk] = ldg8(qp + kk * 16 + h * 8);

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[dt][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  const int total_tiles = (q0 + BQ) / TK;       // key tiles up to the workgroup's last row
  const int nsteps = (total_tiles + 1) / 2;     // steps of the workgroup
  // With 128-key tiles their number can be odd: half 1 then has one tile less (none at all for the first
  // 128 queries) and idles through the last step.
  const int nmine = D == 128 ? nsteps : (total_tiles + 1 - half) / 2;
  // LDS tile = 16 blocks; block b holds rows b, b+16, b+32, b+48 of the tile, 256 bytes each, in
  // the order one wave-wide request delivers them (lane p at +16 p: row b + 16 (p / 16), chunk
  // p % 16 — 16 consecutive lanes fetch one contiguous row), followed by a little padding.  With
  // the padding chosen per operand (K: 16 bytes, V: 64) both kinds of fragment reads are free of
  // bank conflicts, and every fragment address is one per-lane base plus an instruction
  // immediate.  Per half: K tile j in kbuf + (j & 1) tiles, V tile j in vbuf + (j & 1) tiles.
  constexpr uint32_t KBLK = 1024 + 16, VBLK = 1024 + 64, KTILE = 16 * KBLK, VTILE = 16 * VBLK;
  const uint32_t kbuf = (uint32_t)(uintptr_t)(KR_LDS const bf16*)smem + half * 2 * (KTILE + VTILE);
  const uint32_t vbuf = kbuf + 2 * KTILE;
  auto key_of = [&](int j) { return (2 * j + half) * TK; };
  // row-major fragment (K): row 32 t + lane%32, chunk 2 kk + h  ->  + 512 t + 32 kk
  const uint32_t kfrag_lane = (uint32_t)((lane & 15) * KBLK + ((lane >> 4) & 1) * 256 + h * 16);
  // transposed fragment (V): rows 16 g + 4 h + p/4 (+8), channels 32 dt + 16 (lane/16 % 2) +
  // 4 (p % 4)  ->  + 256 g + 64 dt (+ 8 blocks)
  const uint32_t vfrag_lane = (uint32_t)((4 * h + ((lane & 15) >> 2)) * VBLK + ((lane >> 4) & 1) * 32 +
                                         ((lane & 3) >> 1) * 16 + (lane & 1) * 8);

  // One wave requests 4 KiB of a tile: blocks wave + 4 i, i.e. tile rows wave + 4 i (+ 16, 32,
  // 48).  Everything a request needs is kept ready — a pointer to row `wave` of the next tile to
  // ask for, advanced by two tiles per step, the distance of four rows, the lane's byte offset —
  // so that a request costs a handful of scalar instructions: the vector period is bound by the
  // number of instructions the wave has to issue.
  const bf16* kreq = kb + (int64_t)(key_of(0) + wave) * k_ss;
  const bf16* vreq = vb + (int64_t)(key_of(0) + wave) * v_ss;
  const int64_t k_tiles2 = (int64_t)2 * TK * k_ss, v_tiles2 = (int64_t)2 * TK * v_ss;
  const int64_t k_rows4 = 4 * k_ss, v_rows4 = 4 * v_ss;
  const uint32_t k_lane_off = tile_lane_off<D>(lane, (int)k_ss);
  const uint32_t v_lane_off = tile_lane_off<D>(lane, (int)v_ss);
  // one of a tile's four requests of this wave (i = 0..3); the last one moves on to the next tile.  `j` is the
  // tile's step: only the tile a ragged sequence ends in needs it.
  auto request_k_part = [&](uint32_t tile, int j, int i) {
    const uint32_t dst = tile + (wave + 4 * i) * KBLK;
    if (RAGGED && key_of(j) + TK > s)
      request_clamped<D>(kb, k_ss, key_of(j), wave + 4 * i, s, lane, dst);
    else
      dma_b128(kreq + i * k_rows4, k_lane_off, dst);
    if (i == 3) kreq += k_tiles2;
  };
  auto request_v_part = [&](uint32_t tile, int j, int i) {
    const uint32_t dst = tile + (wave + 4 * i) * VBLK;
    if (RAGGED && key_of(j) + TK > s)
      request_clamped<D>(vb, v_ss, key_of(j), wave + 4 * i, s, lane, dst);
    else
      dma_b128(vreq + i * v_rows4, v_lane_off, dst);
    if (i == 3) vreq += v_tiles2;
  };
  auto request_k = [&](uint32_t tile, int j) {
#pragma unroll
    for (int i = 0; i < 4; ++i) request_k_part(tile, j, i);
  };
  auto request_v = [&](uint32_t tile, int j) {
#pragma unroll
    for (int i = 0; i < 4; ++i) request_v_part(tile, j, i);
  };
  // rows of V tile j beyond the sequence: their probabilities are zero, and so must their values be (a copy
  // of the last row could be infinite).  K needs none: masked scores are replaced, whatever they are.
  auto zero_v_tail = [&](int j) {
    if (RAGGED && key_of(j) + TK > s) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        zero_block_tail<D>(key_of(j), wave + 4 * i, s, lane, vbuf + (j & 1) * VTILE + (wave + 4 * i) * VBLK);
    }
  };

  if (D == 128 || nmine > 0) {
    request_k(kbuf, 0);
    if (nmine > 1) request_k(kbuf + KTILE, 1);
    request_v(vbuf, 0);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  if (D == 128 || nmine > 0) zero_v_tail(0);
  kr_barrier();
  if (half == 1) kr_barrier();  // half 1 starts one period late

  bf16x8 pb[NB][2];

  // O^T += V^T . P^T for tile jj of this half (pb holds its probabilities)
  auto pv_step = [&](int jj) {
      uint32_t va = vbuf + (jj & 1) * VTILE + vfrag_lane;
      asm volatile("" : "+v"(va));  // one base register; everything else is an immediate
      auto vfrag = [&](int g, int dt) {  // keys 16 g .. 16 g + 15 of the tile, channels 32 dt ..
        union {
          struct { s16x4 lo, hi; } s;
          bf16x8 v;
        } u;
        const uint32_t a = va + (g & 3) * 256 + (g >> 2) * 128 + dt * 64;
        u.s.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((KR_LDS s16x4*)(a));
        u.s.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((KR_LDS s16x4*)(a + 8 * VBLK));
        return u.v;
      };
      // fragments are fetched one group of four MFMAs ahead, by hand: left to itself the
      // scheduler hoists every read of the period to its start and runs out of registers
      // group g: 16-key groups 4 g / DT .., channel blocks 0 .. DT - 1 of each
      bf16x8 fr[2][4];
#pragma unroll
      for (int u = 0; u < 4; ++u) fr[0][u] = vfrag(u / DT, u % DT);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (g + 1 < 4) {
#pragma unroll
          for (int u = 0; u < 4; ++u) fr[(g + 1) & 1][u] = vfrag((g + 1) * 4 / DT + u / DT, u % DT);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int kg = g * 4 / DT + u / DT;
          oacc[u % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[g & 1][u], pb[kg >> 1][kg & 1],
                                                                 oacc[u % DT], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      };

  settle_scalar_loads();
  for (int j = 0; j < nsteps; ++j) {
    // ---- matrix period: O^T += V^T . P^T of tile j-1, then S^T = K . Q^T of tile j
    f32x16 sacc[NB];
    __builtin_amdgcn_s_setprio(1);
    const bool mine = D == 128 || j < nmine;
    if (j > 0 && (D == 128 || j - 1 < nmine)) pv_step(j - 1);
    if (mine) {
      uint32_t ka = kbuf + (j & 1) * KTILE + kfrag_lane;
      asm volatile("" : "+v"(ka));
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) sacc[t][e] = 0.f;
      auto kfrag = [&](int t, int kk) {
        return *(KR_LDS const bf16x8*)(ka + (t & 1) * 512 + (t >> 1) * 128 + kk * 32);
      };
      bf16x8 fr[2][4];  // group g: contraction steps 2g, 2g+1 for both 32-key blocks
#pragma unroll
      for (int u = 0; u < 4; ++u) fr[0][u] = kfrag(u % NB, u / NB);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (g + 1 < 4) {
#pragma unroll
          for (int u = 0; u < 4; ++u) fr[(g + 1) & 1][u] = kfrag(u % NB, (g + 1) * (4 / NB) + u / NB);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          sacc[u % NB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[g & 1][u], qf[g * (4 / NB) + u / NB],
                                                                 sacc[u % NB], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    kr_barrier();

    // ---- vector period of tile j: the softmax, and between its eight groups of exponentials
    // the eight requests for K(j+2) and V(j+1) (their buffers were last read in the matrix period
    // that just ended).  Issued back to back the requests hold the wave until the address path
    // has taken them, which is as long as the softmax itself.
    const bool want_k = j + 2 < nmine, want_v = j + 1 < nmine;
    const uint32_t k_dst = kbuf + (j & 1) * KTILE, v_dst = vbuf + ((j + 1) & 1) * VTILE;
    if (mine) {
      const int key0 = key_of(j);
      if (key0 + TK - 1 > qw0) {
        asm volatile("" ::: "memory");  // keeps this a branch: off the diagonal no mask code runs
        const int lim = qrow - key0 - 4 * h;  // element offsets beyond it are keys after the query
#pragma unroll
        for (int t = 0; t < NB; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (t * 32 + 8 * (e >> 2) + (e & 3) > lim) sacc[t][e] = -INFINITY;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sacc[t][e]);
      mx = fmaxf(mx, __shfl_xor(mx, 32, KR_WAVE));
      const float m_new = fmaxf(m_run, mx);
      const bool moved = (m_new - m_run) * scale_log2 > kRescaleSlack;  // from -inf: always
      const float m_next = moved ? m_new : m_run;
      const float m_ref = m_next == -INFINITY ? 0.f : m_next;  // nothing seen yet: any finite reference
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_ref) * scale_log2);  // 1 unless moved
      m_run = m_next;
      const float neg_m = -m_ref * scale_log2;
      float psum = 0.f;
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float pe = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[t][e], scale_log2, neg_m));
          psum += pe;
          pb[t][e >> 3][e & 7] = (bf16)pe;
          // eight elements at a time: scheduled freely, all 32 exponent arguments and results
          // would be alive together
          if ((e & 7) == 7) {
            __builtin_amdgcn_sched_barrier(0);
            const int c = t * 2 + (e >> 3);   // 0 .. 2 NB - 1; four of them carry requests
            if (c % (NB / 2) == 0) {
              if (want_k) request_k_part(k_dst, j + 2, c / (NB / 2));
              if (want_v) request_v_part(v_dst, j + 1, c / (NB / 2));
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      l_run = l_run * alpha + psum;
      if (__any(moved)) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int e = 0; e < 16; ++e) oacc[dt][e] *= alpha;
      }
    }
    // what was requested one step ago (K(j+1), V(j)) is read in the next matrix period; exactly
    // the requests of this period (4 per tile and wave, retired in order) may stay in flight
    if (want_k)
      __builtin_amdgcn_s_waitcnt(0x0f78);  // vmcnt(8): K(j+2) and V(j+1) were requested
    else if (want_v)
      __builtin_amdgcn_s_waitcnt(0x0f74);  // vmcnt(4): only V(j+1)
    else
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): nothing was requested
    if (RAGGED && j > 0 && mine) zero_v_tail(j);  // (tile 0 was settled before the loop)
    kr_barrier();
  }
  // last matrix period: the product of the final tile
  __builtin_amdgcn_s_setprio(1);
  if (D == 128 || nsteps - 1 < nmine) pv_step(nsteps - 1);
  __builtin_amdgcn_s_setprio(0);
  kr_barrier();
  if (half == 0) kr_barrier();  // the period half 1 is behind by

  // merge the two halves' partial softmax: half 1 -> LDS -> half 0 (every buffer is idle: the
  // loop ended with a barrier and no request is in flight).  [value][wave][lane] layout.
  float* xch = reinterpret_cast<float*>(smem);
  const int slot = wave * 64 + lane;
  if (half == 1) {
    xch[slot] = m_run;
    xch[256 + slot] = l_run;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) xch[(2 + dt * 16 + e) * 256 + slot] = oacc[dt][e];
  }
  kr_barrier();
  if (half == 1) return;
  {
    const float m_b = xch[slot], l_b = xch[256 + slot];
    const float m_new = fmaxf(m_run, m_b);
    const float a_a = __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2);
    const float a_b = __builtin_amdgcn_exp2f((m_b - m_new) * scale_log2);
    m_run = m_new;
    l_run = l_run * a_a + l_b * a_b;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        oacc[dt][e] = oacc[dt][e] * a_a + xch[(2 + dt * 16 + e) * 256 + slot] * a_b;
  }
  const float l_tot = l_run + __shfl_xor(l_run, 32, KR_WAVE);
  const float inv_l = 1.0f / l_tot;
  RowStage rs;  // behind the (2 + 64) KiB hand-over buffer
  rs.init(reinterpret_cast<char*>(smem) + 68 * 1024 + wave * 4096, lane);
  bf16* op = o + (int64_t)bi * o_sb + kvh * o_sg + hj * o_sh + (int64_t)qw0 * o_ss;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[dt][e] *= inv_l;
  store_rows_bf16<D, RAGGED>(rs, oacc, 1.0f, op, o_ss, s - qw0);
  if (h == 0 && (!RAGGED || qrow < s))
    lse[((int64_t)bi * nq + head) * s + qrow] =
        (m_run * scale_log2 + __builtin_amdgcn_logf(l_tot)) * kLn2;
}

// Ping-pong forward over shared tiles, for launches with enough 256-query tiles to fill the GPU.
// The two halves of four waves own *different* queries (rows 0..127 and 128..255 of the tile) and
// walk the *same* 64-key tiles, half 1 one period behind half 0: a K / V tile is fetched once for
// 256 queries instead of once for 128, there are half as many workgroups to start and to finish,
// and the halves never have to merge anything.  Periods as above: in each, one half feeds the
// matrix pipe (P.V of its previous tile, S = Q.K^T of its next) and the other does its softmax;
// half 0 requests the K tiles during its softmax (K(j+2) while it works on tile j), half 1 the V
// tiles (V(j+2)).  K(j) is read in periods 2j (half 0) and 2j+1 (half 1), V(j) in 2j+2 and 2j+3;
// rings of three tiles each give every request three to four periods to land.  Half 0 needs two
// tiles fewer than half 1 (its rows end 128 earlier) and idles through the last two steps.
template <int D, bool RAGGED>
__global__ __launch_bounds__(512, 1) void attn_fwd_sh_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    bf16* __restrict__ o, float* __restrict__ lse, int s, int nq, int nkv, float scale_log2,
    int64_t q_ss, int64_t q_sb, int64_t q_sg, int64_t q_sh, int64_t k_ss, int64_t k_sb,
    int64_t k_sh, int64_t v_ss, int64_t v_sb, int64_t v_sh, int64_t o_ss, int64_t o_sb,
    int64_t o_sg, int64_t o_sh) {
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];
  constexpr int NB = tile_rows<D> / 32;  // 32-key blocks of a tile
  constexpr int DT = D / 32, KK = D / 16;
  constexpr int TK = tile_rows<D>;       // keys of a tile
  constexpr int BQ2 = 256;

  const int half = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
  const int tid = threadIdx.x & 255;
  const int lane = tid & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nqt = (s + BQ2 - 1) / BQ2;
  int rank, pair;
  longest_first(blockIdx.x, gridDim.x, nqt, rank, pair);
  const int qt = nqt - 1 - rank;
  const int head = pair % nq;
  const int bi = pair / nq;
  const int per = nq / nkv;
  const int kvh = head / per, hj = head % per;

  const int q0 = qt * BQ2;
  const int qw0 = q0 + half * 128 + wave * 32;
  const int qrow = qw0 + (lane & 31);
  const bf16* qp = q + (int64_t)bi * q_sb + kvh * q_sg + hj * q_sh +
                   (int64_t)(RAGGED && qrow >= s ? s - 1 : qrow) * q_ss;
  const bf16* kb = k + (int64_t)bi * k_sb + (int64_t)kvh * k_sh;
  const bf16* vb = v + (int64_t)bi * v_sb + (int64_t)kvh * v_sh;

  bf16x8 qf[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) qf[kk] = ldg8(qp + kk * 16 + h * 8);

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[dt][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  const int ntiles = (q0 + BQ2) / TK;                 // tiles the workgroup walks (>= 2)
  const int nmine = (q0 + half * 128 + 128) / TK;     // tiles with keys this half's rows see
  constexpr uint32_t KBLK = 1024 + 16, VBLK = 1024 + 64, KTILE = 16 * KBLK, VTILE = 16 * VBLK;
  const uint32_t kring = (uint32_t)(uintptr_t)(KR_LDS const bf16*)smem;
  const uint32_t vring = kring + 3 * KTILE;
  const uint32_t kfrag_lane = (uint32_t)((lane & 15) * KBLK + ((lane >> 4) & 1) * 256 + h * 16);
  const uint32_t vfrag_lane = (uint32_t)((4 * h + ((lane & 15) >> 2)) * VBLK + ((lane >> 4) & 1) * 32 +
                                         ((lane & 3) >> 1) * 16 + (lane & 1) * 8);

  // This half's requests: half 0 brings in K tiles, half 1 V tiles; block b of a tile holds its
  // rows b, b + 16, b + 32, b + 48 and wave w fills blocks w + 4 i.  `req` points at row w of the
  // next tile to ask for.
  const int64_t r_ss = half ? v_ss : k_ss;
  const uint32_t r_blk = half ? VBLK : KBLK, r_tile = half ? VTILE : KTILE;
  const uint32_t r_ring = half ? vring : kring;
  const bf16* req = (half ? vb : kb) + (int64_t)wave * r_ss;
  const int64_t r_next = (int64_t)TK * r_ss, r_rows4 = 4 * r_ss;
  const uint32_t r_lane_off = tile_lane_off<D>(lane, (int)r_ss);
  auto request_part = [&](uint32_t tile, int j, int i) {
    const uint32_t dst = tile + (wave + 4 * i) * r_blk;
    if (RAGGED && (j + 1) * TK > s)
      request_clamped<D>(half ? vb : kb, r_ss, j * TK, wave + 4 * i, s, lane, dst);
    else
      dma_b128(req + i * r_rows4, r_lane_off, dst);
    if (i == 3) req += r_next;
  };
  // rows of V tile j (ring slot `slot`) beyond the sequence: as in the kernel above
  auto zero_v_tail = [&](int j, int slot) {
    if (RAGGED && half == 1 && (j + 1) * TK > s) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        zero_block_tail<D>(j * TK, wave + 4 * i, s, lane, vring + slot * VTILE + (wave + 4 * i) * VBLK);
    }
  };
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) request_part(r_ring + t * r_tile, t, i);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  zero_v_tail(0, 0);
  zero_v_tail(1, 1);
  kr_barrier();
  if (half == 1) kr_barrier();  // half 1 starts one period late

  bf16x8 pb[NB][2];

  // O^T += V^T . P^T for the tile in ring slot `slot` (pb holds its probabilities)
  auto pv_step = [&](int slot) {
    uint32_t va = vring + slot * VTILE + vfrag_lane;
    asm volatile("" : "+v"(va));
    auto vfrag = [&](int g, int dt) {
      union {
        struct { s16x4 lo, hi; } s;
        bf16x8 v;
      } u;
      const uint32_t a = va + (g & 3) * 256 + (g >> 2) * 128 + dt * 64;
      u.s.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((KR_LDS s16x4*)(a));
      u.s.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((KR_LDS s16x4*)(a + 8 * VBLK));
      return u.v;
    };
    bf16x8 fr[2][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) fr[0][u] = vfrag(u / DT, u % DT);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (g + 1 < 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u) fr[(g + 1) & 1][u] = vfrag((g + 1) * 4 / DT + u / DT, u % DT);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int kg = g * 4 / DT + u / DT;
        oacc[u % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[g & 1][u], pb[kg >> 1][kg & 1],
                                                               oacc[u % DT], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  int slot = 0, slot_prev = 2, slot_req = 2;  // j % 3, (j - 1) % 3, (j + 2) % 3
  settle_scalar_loads();
  for (int j = 0; j < ntiles; ++j) {
    // ---- matrix period: O^T += V^T . P^T of tile j-1, then S^T = K . Q^T of tile j
    f32x16 sacc[NB];
    const bool mine = j < nmine;
    __builtin_amdgcn_s_setprio(1);
    if (j > 0 && j - 1 < nmine) pv_step(slot_prev);
    if (mine) {
      uint32_t ka = kring + slot * KTILE + kfrag_lane;
      asm volatile("" : "+v"(ka));
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) sacc[t][e] = 0.f;
      auto kfrag = [&](int t, int kk) {
        return *(KR_LDS const bf16x8*)(ka + (t & 1) * 512 + (t >> 1) * 128 + kk * 32);
      };
      bf16x8 fr[2][4];
#pragma unroll
      for (int u = 0; u < 4; ++u) fr[0][u] = kfrag(u % NB, u / NB);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (g + 1 < 4) {
#pragma unroll
          for (int u = 0; u < 4; ++u) fr[(g + 1) & 1][u] = kfrag(u % NB, (g + 1) * (4 / NB) + u / NB);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          sacc[u % NB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[g & 1][u], qf[g * (4 / NB) + u / NB],
                                                                 sacc[u % NB], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    kr_barrier();

    // ---- vector period of tile j: the softmax, and between its four groups of exponentials
    // this wave's four requests for tile j+2 of its operand (the ring slot was last read two
    // periods ago).  Half 0 has no request left once it has run out of tiles of its own.
    const bool want = j + 2 < ntiles;
    const uint32_t r_dst = r_ring + slot_req * r_tile;
    if (mine) {
      const int key0 = j * TK;
      if (key0 + TK - 1 > qw0) {
        asm volatile("" ::: "memory");  // keeps this a branch: off the diagonal no mask code runs
        const int lim = qrow - key0 - 4 * h;  // element offsets beyond it are keys after the query
#pragma unroll
        for (int t = 0; t < NB; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (t * 32 + 8 * (e >> 2) + (e & 3) > lim) sacc[t][e] = -INFINITY;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sacc[t][e]);
      mx = fmaxf(mx, __shfl_xor(mx, 32, KR_WAVE));
      const float m_new = fmaxf(m_run, mx);
      const bool moved = (m_new - m_run) * scale_log2 > kRescaleSlack;  // from -inf: always
      const float m_next = moved ? m_new : m_run;
      const float m_ref = m_next == -INFINITY ? 0.f : m_next;
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_ref) * scale_log2);  // 1 unless moved
      m_run = m_next;
      const float neg_m = -m_ref * scale_log2;
      float psum = 0.f;
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float pe = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[t][e], scale_log2, neg_m));
          psum += pe;
          pb[t][e >> 3][e & 7] = (bf16)pe;
          if ((e & 7) == 7) {
            __builtin_amdgcn_sched_barrier(0);
            const int c = t * 2 + (e >> 3);
            if (c % (NB / 2) == 0 && want) request_part(r_dst, j + 2, c / (NB / 2));
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      l_run = l_run * alpha + psum;
      if (__any(moved)) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int e = 0; e < 16; ++e) oacc[dt][e] *= alpha;
      }
    } else if (want) {
#pragma unroll
      for (int i = 0; i < 4; ++i) request_part(r_dst, j + 2, i);
    }
    // tile j+1 of this half's operand (requested one step ago) is read from the next period on;
    // only this period's four requests may stay in flight
    if (want)
      __builtin_amdgcn_s_waitcnt(0x0f74);  // vmcnt(4)
    else
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    if (RAGGED && j > 0 && j + 1 < ntiles) zero_v_tail(j + 1, slot == 2 ? 0 : slot + 1);
    kr_barrier();
    slot_prev = slot;
    slot = slot == 2 ? 0 : slot + 1;
    slot_req = slot_req == 2 ? 0 : slot_req + 1;
  }
  // last matrix period: the product of the final tile (half 1; half 0 finished two steps ago)
  if (ntiles - 1 < nmine) {
    __builtin_amdgcn_s_setprio(1);
    pv_step(slot_prev);
    __builtin_amdgcn_s_setprio(0);
  }
  if (half == 0) kr_barrier();  // the barrier half 1 spent on starting late

  // No tile is requested any more and K tiles are no longer read: each wave stages its output
  // rows through 4 KiB of the K ring.
  const float l_tot = l_run + __shfl_xor(l_run, 32, KR_WAVE);
  const float inv_l = 1.0f / l_tot;
  RowStage rs;
  rs.init(reinterpret_cast<char*>(smem) + (half * 4 + wave) * 4096, lane);
  bf16* op = o + (int64_t)bi * o_sb + kvh * o_sg + hj * o_sh + (int64_t)qw0 * o_ss;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[dt][e] *= inv_l;
  store_rows_bf16<D, RAGGED>(rs, oacc, 1.0f, op, o_ss, s - qw0);
  if (h == 0 && (!RAGGED || qrow < s))
    lse[((int64_t)bi * nq + head) * s + qrow] =
        (m_run * scale_log2 + __builtin_amdgcn_logf(l_tot)) * kLn2;
}

// delta and the log2-domain statistics have rows of sp = s rounded up to 128: positions beyond s get values
// that make their probabilities exactly zero.
constexpr float kPadLse = 1e30f;  // exp2(x - 1.4e30) = 0 for every finite score

template <int D>
__global__ __launch_bounds__(256) void attn_delta_kernel(const bf16* __restrict__ dout,
                                                         const bf16* __restrict__ o,
                                                         const float* __restrict__ lse,
                                                         float* __restrict__ neg_delta,
                                                         float* __restrict__ neg_lse2, int s, int sp, int nq,
                                                         int per, int64_t total_rows, QLayout dol,
                                                         QLayout ol) {
  constexpr int LPR = D / 8;  // lanes per (batch, head, position) row
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LPR;
  const int sub = threadIdx.x & (LPR - 1);
  if (row >= total_rows) return;
  const int si = (int)(row % sp);
  const int head = (int)((row / sp) % nq);
  const int bi = (int)(row / ((int64_t)sp * nq));
  if (si >= s) {
    if (sub == 0) {
      neg_delta[row] = 0.f;
      neg_lse2[row] = -kPadLse * kLog2e;
    }
    return;
  }
  const bf16x8 a = ldg8(dout + dol.at(bi, head, per) + (int64_t)si * dol.s_ + sub * 8);
  const bf16x8 b = ldg8(o + ol.at(bi, head, per) + (int64_t)si * ol.s_ + sub * 8);
  float acc = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) acc += (float)a[e] * (float)b[e];
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, KR_WAVE);
  if (sub == 0) {
    neg_delta[row] = -acc;
    // -lse in the log2 domain, so that the dK/dV kernel's exponent is one multiply-add and its
    // row statistics can go straight from global memory into LDS
    neg_lse2[row] = -lse[((int64_t)bi * nq + head) * s + si] * kLog2e;
  }
}

// dK/dV with the waves of a SIMD specialised.  A wave issues at most one instruction every 4-5
// cycles, and one wave that does everything for its 32 keys (scores, exponentials, both
// accumulating products) needs 128 accumulator and 64 K/V-fragment registers — no room for a
// second wave on the SIMD — so it is bound by that rate: 850 instructions per 64 MFMAs.  Instead
// a workgroup has eight waves, two per SIMD, for its 128 keys:
//   waves 0-3 ("score" waves, 32 keys each, K and V fragments in registers) compute S = Q.K^T and
//     dP = dO.V^T of a 32-query block, P and dS from them, and hand P, dS (bf16, already in the
//     B-operand layout of the next products) to their partner through 4 KB of LDS;
//   waves 4-7 ("accumulate" waves, the partner on the same SIMD) hold dK and dV and issue
//     dV^T += dO^T.P and dK^T += Q^T.dS with the Q / dO tiles read transposed; they also issue
//     every global -> LDS request, which keeps the score waves' instruction stream short.
// Both run well below 256 registers, so the matrix products write plain VGPRs (no accumulator
// copies).  Two barriers per 64-query tile: after each, the accumulate waves pick up the block
// the score waves finished before it, so the two kinds of work overlap with one block of lag.
// Three LDS stages: tile it is read as rows by the score waves and transposed by the accumulate
// waves; every read of it is issued before the second barrier of iteration it, so tile it+3 is
// requested right after that barrier into the same stage and has an iteration and a half to
// land (it must be complete by the first barrier of iteration it+2: the score waves start on a
// tile one block ahead).
// PARTIAL = true: fp32 results for this query head go to part_k / part_v [b, nq, qsplit, sp, D].
// (Head dimension 128; attn_bwd_dkdv64_kernel below takes 64.)
template <bool RAGGED, bool PARTIAL>
__global__ __launch_bounds__(512, 1) void attn_bwd_dkdv_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    const bf16* __restrict__ dout, const float* __restrict__ neg_lse2, const float* __restrict__ neg_delta,
    bf16* __restrict__ dk, bf16* __restrict__ dv, float* __restrict__ part_k,
    float* __restrict__ part_v, int s, int nq, int nkv, int qsplit, int hpw, float scale, float scale_log2,
    QLayout ql, KLayout kl, KLayout vl, QLayout dol, KLayout dkl, KLayout dvl) {
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];
  constexpr int D = HD, TQ = tile_rows<D>;  // queries of a tile: two blocks of 32
  constexpr int DT = D / 32, KK = D / 16;
  constexpr int NF = 4 * DT;                        // transposed fragments of a block, two channel operands
  // stage layout: Q tile | dO tile (blocked tiles) | -lse[TQ] fp32 | -delta[TQ] fp32
  constexpr uint32_t STAGE = 2 * BT_BYTES + 8 * TQ;  // bytes
  constexpr int NS = 3;
  // hand-over area behind the stages: [block parity][key block][slot 0..3][lane] 16 bytes each
  constexpr uint32_t XCH = NS * STAGE;

  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
  const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int role = wave8 >> 2;  // 0: score wave, 1: accumulate wave
  const int wave = wave8 & 3;   // key block of the tile
  const int sp = RAGGED ? (s + 127) / 128 * 128 : s;  // rows of the statistics and of the partial results
  const int nkt = sp / 128;
  // (a key tile's parts count as tiles of half its length; low key tiles see the most queries)
  int rank, hg;
  longest_first(blockIdx.x, gridDim.x, nkt * qsplit, rank, hg);
  const int part = rank % qsplit, kt = rank / qsplit;
  // A workgroup takes `hpw` consecutive query heads of one KV group, one after the other: its K / V
  // fragments and its dK / dV accumulators serve them all, so a group leaves per / hpw partial
  // results instead of per (none at all when hpw = per), and the workgroup's start and end are
  // paid once for hpw heads.  The host picks hpw so that enough workgroups remain.
  const int nhg = nq / hpw;
  const int hgroup = hg % nhg;
  const int head = hgroup * hpw;  // the first of this workgroup's heads
  const int bi = hg / nhg;
  const int per = nq / nkv;
  const int kvh = head / per;
  const int key0 = kt * 128;
  const int kw0 = key0 + wave * 32;
  const int krow = kw0 + (lane & 31);
  const int qt_first = key0 / TQ;
  // this part's query tiles, per head
  const int niter = (sp / TQ - qt_first - part + qsplit - 1) / qsplit;
  const int nit_all = niter * hpw;                                       // ... over all heads of the workgroup
  const uint32_t lds0 = (uint32_t)(uintptr_t)(KR_LDS const bf16*)smem;
  const uint32_t xch_lane = lds0 + XCH + wave * 4096 + lane * 16;  // + parity * 16384 + slot * 1024

  if (role == 0) {
    // ------------------------------------------------------------------ score waves
    const bf16* kp = k + kl.at(bi, kvh) + (int64_t)(RAGGED && krow >= s ? s - 1 : krow) * kl.s_;
    const bf16* vp = v + vl.at(bi, kvh) + (int64_t)(RAGGED && krow >= s ? s - 1 : krow) * vl.s_;
    bf16x8 kf[KK], vf[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      kf[kk] = ldg8(kp + kk * 16 + h * 8);
      vf[kk] = ldg8(vp + kk * 16 + h * 8);
    }
    kr_barrier();  // tile 0 (and 1) requested by the accumulate waves have landed
    // S = Q.K^T and dP = dO.V^T of one 32-query block: sixteen fragments, then sixteen MFMAs
    auto issue_scores = [&](int stage, int sub, f32x16& sacc, f32x16& dpacc) {
      uint32_t q_rows = lds0 + stage * STAGE + bt_rows_lane(lane);
      uint32_t do_rows = q_rows + BT_BYTES;
      asm volatile("" : "+v"(q_rows), "+v"(do_rows));  // one base register each; the rest are immediates
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        sacc[e] = 0.f;
        dpacc[e] = 0.f;
      }
      bf16x8 qfr[KK], dofr[KK];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        qfr[kk] = bt_rows<D>(q_rows, sub, kk);
        dofr[kk] = bt_rows<D>(do_rows, sub, kk);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qfr[kk], kf[kk], sacc, 0, 0, 0);
        dpacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dofr[kk], vf[kk], dpacc, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    // One step: P = exp2(S c - lse), dS = P (dP - delta) of block (stage, sub), handed to the
    // partner wave, while the score products of the block after it (nstage, nsub) are issued.
    // A wave's instructions issue in order and an MFMA waits for the matrix pipe, so sixteen
    // MFMAs in a row stall the wave for as long as they take; four at a time between the four
    // groups of exponentials they cost (almost) nothing.
    auto step = [&](int stage, int sub, int qs0, f32x16& sacc, const f32x16& dpacc, int nstage, int nsub,
                    f32x16& nsacc, f32x16& ndpacc) {
      const float* stats = reinterpret_cast<const float*>(reinterpret_cast<const char*>(smem) +
                                                          stage * STAGE + 2 * BT_BYTES);
      uint32_t q_rows = lds0 + nstage * STAGE + bt_rows_lane(lane);
      uint32_t do_rows = q_rows + BT_BYTES;
      asm volatile("" : "+v"(q_rows), "+v"(do_rows));
      bf16x8 qfr[KK], dofr[KK];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        qfr[kk] = bt_rows<D>(q_rows, nsub, kk);
        dofr[kk] = bt_rows<D>(do_rows, nsub, kk);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        nsacc[e] = 0.f;
        ndpacc[e] = 0.f;
      }
      // lane: key column krow, query rows qs0 + 8g + 4h + e; only blocks that reach the diagonal
      // pay for the causal mask
      if (qs0 < kw0 + 31) {
        const int lim = krow - qs0 - 4 * h;  // element offsets below it are queries before the key
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          float x = 8 * (e >> 2) + (e & 3) < lim ? -INFINITY : sacc[e];
          asm volatile("" : "+v"(x));  // keeps this a branch: off the diagonal no mask code runs
          sacc[e] = x;
        }
      }
      bf16x8 pb[2], dsb[2];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 l4 = *reinterpret_cast<const f32x4*>(stats + sub * 32 + 8 * g + 4 * h);
        const f32x4 d4 = *reinterpret_cast<const f32x4*>(stats + TQ + sub * 32 + 8 * g + 4 * h);
#pragma unroll
        for (int kk = g * KK / 4; kk < (g + 1) * KK / 4; ++kk) {
          nsacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qfr[kk], kf[kk], nsacc, 0, 0, 0);
          ndpacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dofr[kk], vf[kk], ndpacc, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[g * 4 + e], scale_log2, l4[e]));
          const float ds = p * (dpacc[g * 4 + e] + d4[e]);
          pb[g >> 1][(g & 1) * 4 + e] = (bf16)p;
          dsb[g >> 1][(g & 1) * 4 + e] = (bf16)ds;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      const uint32_t xa = xch_lane + (sub & 1) * 16384;
      *(KR_LDS bf16x8*)(xa) = pb[0];
      *(KR_LDS bf16x8*)(xa + 1024) = pb[1];
      *(KR_LDS bf16x8*)(xa + 2048) = dsb[0];
      *(KR_LDS bf16x8*)(xa + 3072) = dsb[1];
    };
    // The score products of a block are thus issued one block ahead of the exponentials that
    // consume them (the first block of the next tile during the second block of this one: that
    // tile is complete by the first barrier of the iteration; behind the last tile a stale
    // stage is read, unused).
    f32x16 s0, dp0, s1, dp1;
    settle_scalar_loads();
    issue_scores(0, 0, s0, dp0);
    for (int it = 0, itl = 0; it < nit_all; ++it) {
      const int stage = it % NS;
      const int q0 = (qt_first + itl * qsplit + part) * TQ;
      itl = itl + 1 == niter ? 0 : itl + 1;  // the next head starts over at the diagonal
      step(stage, 0, q0, s0, dp0, stage, 1, s1, dp1);
      kr_barrier();  // hand-over of block 0
      step(stage, 1, q0 + 32, s1, dp1, (it + 1) % NS, 0, s0, dp0);
      kr_barrier();  // hand-over of block 1
    }
    return;
  }

  // -------------------------------------------------------------------- accumulate waves
  const bf16* qb = q + ql.at(bi, head, per);
  const bf16* dob = dout + dol.at(bi, head, per);
  const int64_t stat0 = ((int64_t)bi * nq + head) * sp;
  // A tile is brought in by nine requests per wave (eight for waves 2 and 3): the TQ + TQ row
  // statistics, 4 bytes per lane, 64 of them per wave, then four consecutive rows (+ 16, 32, 48
  // through the lanes) of the Q tile and four of the dO tile.  request_begin names the tile,
  // request_piece(i) issues piece i = 0..8, in this order (requests retire in order).
  uint32_t req_tile = 0, req_lane_off = 0;
  const bf16* req_row = nullptr;
  const bf16 *req_q = qb, *req_do = dob;
  int64_t req_stat = stat0;
  int req_qt = 0;
  const bool has_stat = wave < 2;
  auto request_begin = [&](int it) {
    const int hh = it / niter, itl = it - hh * niter;  // head of the workgroup, query tile of that head
    req_qt = qt_first + itl * qsplit + part;
    req_tile = lds0 + (it % NS) * STAGE;
    req_q = qb + hh * ql.h_;    // consecutive heads of one KV group
    req_do = dob + hh * dol.h_;
    req_stat = stat0 + (int64_t)hh * sp;
  };
  auto request_piece = [&](int i) {
    if (i == 0) {
      if (has_stat) {
        int l2 = lane;
        asm volatile("" : "+v"(l2));
        dma_b32((wave == 0 ? neg_lse2 : neg_delta) + req_stat + req_qt * TQ, (uint32_t)l2 * 4u,
                req_tile + 2 * BT_BYTES + wave * 256);
      }
      return;
    }
    const int j = (i - 1) & 3;
    const bool second = i > 4;
    if (RAGGED && (req_qt + 1) * TQ > s) {  // the tile the sequence ends in
      request_clamped<D>(second ? req_do : req_q, second ? dol.s_ : ql.s_, req_qt * TQ, 4 * wave + j, s, lane,
                         req_tile + (second ? BT_BYTES : 0) + (wave + 4 * j) * BT_BLK);
      return;
    }
    if (j == 0) {
      int l2 = lane;
      asm volatile("" : "+v"(l2));  // the lane offset lives only across the four requests of a tile
      const int64_t ss = second ? dol.s_ : ql.s_;
      req_lane_off = tile_lane_off<D>(l2, (int)ss);
      req_row = (second ? req_do : req_q) + ((int64_t)req_qt * TQ + 4 * wave) * ss;
    }
    dma_b128(req_row, req_lane_off, req_tile + (second ? BT_BYTES : 0) + (wave + 4 * j) * BT_BLK);
    req_row += second ? dol.s_ : ql.s_;
  };
  auto request_tile = [&](int it) {
    request_begin(it);
#pragma unroll
    for (int i = 0; i < 9; ++i) request_piece(i);
  };
  // wait until at most the requests of one tile (the newest) are in flight
  auto wait_all_but_newest_tile = [&]() {
    if (has_stat)
      __builtin_amdgcn_s_waitcnt(0x0f79);  // vmcnt(9)
    else
      __builtin_amdgcn_s_waitcnt(0x0f78);  // vmcnt(8)
  };
  // zeros in the rows of iteration it's tile that lie beyond the sequence, once its requests have landed: their
  // probabilities are zero (see kPadLse), and so must the factors be
  auto zero_tail = [&](int it) {
    if (RAGGED && it < nit_all) {
      const int row0 = (qt_first + (it % niter) * qsplit + part) * TQ;
      if (row0 + TQ > s) {
        const uint32_t tile = lds0 + (it % NS) * STAGE;
        bt_zero_tail<D>(row0, s, tile, wave, lane);
        bt_zero_tail<D>(row0, s, tile + BT_BYTES, wave, lane);
      }
    }
  };
  f32x16 dkacc[DT], dvacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      dkacc[dt][e] = 0.f;
      dvacc[dt][e] = 0.f;
    }
  request_tile(0);
  if (nit_all > 1) request_tile(1);
  if (nit_all > 2) {
    request_tile(2);
    wait_all_but_newest_tile();
  } else {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  }
  zero_tail(0);
  zero_tail(1);
  kr_barrier();
  // The transposed fragments of a block (fr[2 DT k2 + 2 dt]: dO^T, fr[2 DT k2 + 2 dt + 1]: Q^T,
  // queries 16 k2 .. of the block, channels 32 dt ..) live in registers across blocks: each is
  // refilled for the next block right behind the MFMA that consumed it (one MFMA later), so the
  // LDS reads of the next block ride under this block's matrix work and the wave reaches the
  // next barrier with its operands already there.
  const uint32_t cols_lane = bt_cols_lane(lane);
  auto frag = [&](uint32_t stage_base, int sub, int f) {
    const uint32_t base = stage_base + ((f & 1) ? 0u : BT_BYTES);  // odd: Q tile, even: dO tile
    return bt_cols<D>(base, 2 * sub + f / (2 * DT), (f >> 1) % DT);
  };
  bf16x8 fr[NF];
  {
    uint32_t base = lds0 + cols_lane;
    asm volatile("" : "+v"(base));
#pragma unroll
    for (int f = 0; f < NF; ++f) fr[f] = frag(base, 0, f);
  }
  settle_scalar_loads();
  for (int it = 0; it < nit_all; ++it) {
    const int stage = it % NS;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      // tile it+1 (requested an iteration and a half ago) must have landed before this
      // iteration's first barrier: the score waves start on it right after.  Tile it+2 may still
      // be on its way.
      if (sub == 0 && it > 0) {  // (tiles 0 and 1 were awaited before the loop)
        if (it + 2 < nit_all) {
          // in flight behind tile it+1: the first five pieces of tile it+2
          if (has_stat)
            __builtin_amdgcn_s_waitcnt(0x0f75);  // vmcnt(5)
          else
            __builtin_amdgcn_s_waitcnt(0x0f74);  // vmcnt(4)
        } else {
          __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        }
        zero_tail(it + 1);
      }
      kr_barrier();
      // After the last barrier nobody reads tile it any more (this wave fetched its last
      // fragments of it during the block before, the score waves before the barrier in front of this):
      // tile it+3 goes into its stage, one request behind each of the first MFMAs — pieces 0-4
      // in this block, pieces 5-8 in the first block of the next iteration, so that neither
      // block of the accumulate waves outlasts the score waves' step beside it.
      const bool first_pieces = sub == 1 && it + 3 < nit_all;
      const bool last_pieces = sub == 0 && it > 0 && it + 2 < nit_all;
      if (first_pieces) request_begin(it + 3);
      const uint32_t xa = xch_lane + (sub & 1) * 16384;
      bf16x8 hand[4];  // P (queries 0-15, 16-31 of the block), dS (the same)
#pragma unroll
      for (int c = 0; c < 4; ++c) hand[c] = *(KR_LDS const bf16x8*)(xa + c * 1024);
      // next block: the next of this tile, or the first of the next tile (complete since this
      // iteration's first barrier; behind the last tile a stale stage, unused)
      uint32_t next_base = lds0 + (sub == 0 ? stage : (it + 1) % NS) * STAGE + cols_lane;
      asm volatile("" : "+v"(next_base));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const int dt = (f >> 1) % DT;
        if (f & 1)
          dkacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[f], hand[2 + f / (2 * DT)], dkacc[dt], 0, 0, 0);
        else
          dvacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[f], hand[f / (2 * DT)], dvacc[dt], 0, 0, 0);
        if (f > 0) fr[f - 1] = frag(next_base, sub ^ 1, f - 1);
        if (first_pieces && f < 5) request_piece(f);
        if (last_pieces && f < 4) request_piece(5 + f);
        __builtin_amdgcn_sched_barrier(0);
      }
      fr[NF - 1] = frag(next_base, sub ^ 1, NF - 1);
    }
  }

  // The hand-over slice this wave read last is its own: use the other one (block parity 0, read
  // one barrier earlier by this wave only) for the output transposition.
  RowStage rs;
  rs.init(reinterpret_cast<char*>(smem) + XCH + wave * 4096, lane);
  if (PARTIAL) {
    const int64_t prow = (((int64_t)bi * nhg + hgroup) * qsplit + part) * sp + kw0;
    store_rows_f32<D>(rs, dkacc, scale, part_k + prow * D, D);
    store_rows_f32<D>(rs, dvacc, 1.0f, part_v + prow * D, D);
  } else {
    store_rows_bf16<D, RAGGED>(rs, dkacc, scale, dk + dkl.at(bi, kvh) + (int64_t)kw0 * dkl.s_, dkl.s_, s - kw0);
    store_rows_bf16<D, RAGGED>(rs, dvacc, 1.0f, dv + dvl.at(bi, kvh) + (int64_t)kw0 * dvl.s_, dvl.s_, s - kw0);
  }
}
// dK/dV at head dimension 64.  A wave's K and V fragments and both accumulators are half of what 128 channels take
// (96 registers instead of 192), so a wave does all the work of its 32 keys — scores, exponentials, both accumulating
// products — and no hand-over is needed.  Eight waves, two per SIMD: waves w and w + 4 have the same 32 of the
// workgroup's 128 keys and take the first and the second 64 queries of every 128-query tile; at the end one of them
// gets the sum of dK, the other of dV.  Four stages of a Q and a dO tile, one barrier per tile.
// The loop is one pipeline of sixteen slots per 32-query block b, each slot one MFMA (32 cycles of the matrix pipe) and
// the vector work of one score (multiply-add, exponential, multiplication, conversions: 27 cycles), so that one
// wave alone already keeps the pipe nearly full:
//   slots 0-7    S and dP of block b + 1
//   slots 8-11   dV and dK, first 16 queries of block b
//   slots 12-15  ... last 16 queries
// A score's multiply-add, its exponential and its remaining work are in consecutive slots (in one slot a wave would wait for
// each of them); score 0 of block b + 1 starts in slot 10 of block b.
// What bounds it: no unit alone.  The matrix pipes are busy 58 % of the cycles, the vector ALUs 47, the LDS pipes 59, a wave waits a
// quarter of its time, and the power limit leaves 1.8 of 2.4 GHz; without LDS reads, requests and barriers it takes 203 us where it
// takes 274.  The kernel that specialised its waves, as the one above does, waited for hand-overs: b 2 x 32/8 x s 4096 404 -> 274 us
// (0.70 -> 1.03 PFLOP/s of the four products), b 1 beside other streams 199 -> 143, s 2048, b 1 60 -> 46, 4 x 1000 tokens, 8 heads 38
// (with the sum of its partial results) -> 22.  Short rows pay for the exchange at the end: s 256, 8/8 heads 11.8 (with that sum) ->
// 9.2, 8/2 heads 12.4 -> 13.5.
// Two independent workgroups of four waves per compute unit took 309 (each a barrier fewer, but the first key tiles
// run on alone); row statistics through one lane each and lane broadcasts, instead of 8 KB of LDS reads a block, the same.
// Everything read from LDS is requested about four slots before it is used.  dP starts from -delta, read straight into
// the accumulator, which takes the subtraction out of every score.
// PARTIAL = true: fp32 results for this group of heads go to part_k / part_v [b, nq / hpw, qsplit, sp, 64].
template <bool RAGGED, bool PARTIAL>
__global__ __launch_bounds__(512, 1) void attn_bwd_dkdv64_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    const bf16* __restrict__ dout, const float* __restrict__ neg_lse2, const float* __restrict__ neg_delta,
    bf16* __restrict__ dk, bf16* __restrict__ dv, float* __restrict__ part_k,
    float* __restrict__ part_v, int s, int nq, int nkv, int qsplit, int hpw, float scale, float scale_log2,
    QLayout ql, KLayout kl, KLayout vl, QLayout dol, KLayout dkl, KLayout dvl) {
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];
  constexpr int D = 64, TQ = tile_rows<D>, DT = D / 32, KK = D / 16;
  constexpr uint32_t STAGE = 2 * BT_BYTES + 8 * TQ;  // Q tile | dO tile | -lse[TQ] fp32 | -delta[TQ] fp32
  constexpr int NS = 4;

  const int lane = threadIdx.x & 63, h = lane >> 5;
  const int wave8 = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wave = wave8 & 3, half = wave8 >> 2;  // key block of the tile; which 64 queries of a tile
  const int sp = RAGGED ? (s + 127) / 128 * 128 : s;  // rows of the statistics and of the partial results
  const int nkt = sp / 128;
  int rank, hg;
  longest_first(blockIdx.x, gridDim.x, nkt * qsplit, rank, hg);
  const int part = rank % qsplit, kt = rank / qsplit;  // low key tiles see the most queries
  const int nhg = nq / hpw;
  const int hgroup = hg % nhg;
  const int head = hgroup * hpw;  // `hpw` consecutive query heads of one KV group, one after the other
  const int bi = hg / nhg;
  const int per = nq / nkv;
  const int kvh = head / per;
  const int kw0 = kt * 128 + wave * 32;
  const int krow = kw0 + (lane & 31);
  const int kld = RAGGED && krow >= s ? s - 1 : krow;
  const int niter = (nkt - kt - part + qsplit - 1) / qsplit;  // this part's query tiles, per head
  const int nit_all = niter * hpw;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(KR_LDS const bf16*)smem;

  const bf16* kp = k + kl.at(bi, kvh) + (int64_t)kld * kl.s_;
  const bf16* vp = v + vl.at(bi, kvh) + (int64_t)kld * vl.s_;
  bf16x8 kf[KK], vf[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    kf[kk] = ldg8(kp + kk * 16 + h * 8);
    vf[kk] = ldg8(vp + kk * 16 + h * 8);
  }

  // A tile is brought in by the eight waves together: waves 0-3 request 64 of its row statistics each (0, 1: -lse, 2, 3:
  // -delta), then every wave two blocks of the Q tile and two of the dO tile (block B of a tile holds its rows r, r + 16, r +
  // 32, r + 48, r = 4 (B % 4) + B / 4, and + 64): blocks wave8 and wave8 + 8, rows r0 and r0 + 2.  Pointers to row r0 of
  // the next tile are kept, so that a request is a handful of scalar instructions.
  const int r0 = 4 * wave + half;
  const bf16* qb = q + ql.at(bi, head, per);
  const bf16* dob = dout + dol.at(bi, head, per);
  const float* statb = (wave < 2 ? neg_lse2 : neg_delta) + ((int64_t)bi * nq + head) * sp + (wave & 1) * 64;
  const uint32_t q_lane = tile_lane_off<D>(lane, (int)ql.s_), do_lane = tile_lane_off<D>(lane, (int)dol.s_);
  const uint32_t stat_lane4 = (uint32_t)lane * 4u;
  const int64_t q_step = (int64_t)(qsplit * TQ) * ql.s_, do_step = (int64_t)(qsplit * TQ) * dol.s_;
  int req_it = 0, req_head = 0, req_qt = kt + part;  // the next tile to ask for
  const bf16 *q_next = nullptr, *do_next = nullptr;
  const float* stat_next = nullptr;
  auto seek = [&]() {
    q_next = qb + req_head * ql.h_ + (int64_t)(req_qt * TQ + r0) * ql.s_;
    do_next = dob + req_head * dol.h_ + (int64_t)(req_qt * TQ + r0) * dol.s_;
    stat_next = statb + (int64_t)req_head * sp + req_qt * TQ;
  };
  seek();
  // One piece of the next tile (0: statistics, which both halves ask for, 1, 2: Q, 3, 4: dO).  Behind the last tile that one
  // is asked for again, into a free stage: no branch, so that the pipeline below stays one block of code.
  auto request_piece = [&](uint32_t stage, int i) {
    const int j = (i - 1) & 1;
    const bool second = i > 2;
    const uint32_t dst = stage + (second ? BT_BYTES : 0) + (wave8 + 8 * j) * BT_BLK;
    if (i == 0)
      dma_b32(stat_next, stat_lane4, stage + 2 * BT_BYTES + wave * 256);
    else if (RAGGED)
      request_clamped<D>(second ? dob + req_head * dol.h_ : qb + req_head * ql.h_, second ? dol.s_ : ql.s_, req_qt * TQ,
                         r0 + 2 * j, s, lane, dst);
    else if (second)
      dma_b128(do_next + 2 * j * dol.s_, do_lane, dst);
    else
      dma_b128(q_next + 2 * j * ql.s_, q_lane, dst);
  };
  auto requested = [&]() {  // on to the next tile; the next head starts over at the diagonal
    if (++req_it >= nit_all) return;
    req_qt += qsplit;
    if (req_qt >= nkt) {
      req_qt = kt + part;
      ++req_head;
      seek();
    } else {
      q_next += q_step;
      do_next += do_step;
      stat_next += qsplit * TQ;
    }
  };
  // rows of query tile qt beyond the sequence: zeros once they have landed (their probabilities are zero, see kPadLse)
  auto zero_tail = [&](uint32_t stage, int qt) {
    if (RAGGED && (qt + 1) * TQ > s) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        zero_block_tail<D>(qt * TQ, r0 + 2 * j, s, lane, stage + (wave8 + 8 * j) * BT_BLK);
        zero_block_tail<D>(qt * TQ, r0 + 2 * j, s, lane, stage + BT_BYTES + (wave8 + 8 * j) * BT_BLK);
      }
    }
  };
  f32x16 dkacc[DT], dvacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      dkacc[dt][e] = 0.f;
      dvacc[dt][e] = 0.f;
    }
  const uint32_t rows_lane = bt_rows_lane(lane), cols_lane = bt_cols_lane(lane) + half * 128;
  const uint32_t rows_half = rows_lane + half * 128;  // 32-row blocks 2 and 3 are column half 1 of the tile's image
  const uint32_t stat_lane = 2 * BT_BYTES + 16 * h + half * 256;

  struct Scores { f32x16 s, dp; };
  bf16x8 qfr[3], dofr[3];      // row fragments, contraction step kk in place kk % 3
  bf16x8 fr[2 * DT];           // transposed fragments: dO^T, Q^T of each channel block
  f32x4 l4[2];                 // -lse of four scores, group g in place g % 2
  u32x4 pb[2], dsb[2];         // P and dS of the block, rounded to bf16, two to a register
  float x_at = 0.f, p_at = 0.f, p_even = 0.f, ds_even = 0.f;  // scores under way
  auto row_frag = [&](uint32_t rows, int sub, int kk) {
    qfr[kk % 3] = bt_rows<D>(rows, sub, kk);
    dofr[kk % 3] = bt_rows<D>(rows + BT_BYTES, sub, kk);
  };
  auto begin_dp = [&](Scores& x, uint32_t stats, int sub, int g) {
    const f32x4 d4 = *(KR_LDS const f32x4*)(stats + 4 * (TQ + sub * 32 + 8 * g));
#pragma unroll
    for (int e = 0; e < 4; ++e) x.dp[4 * g + e] = d4[e];
  };
  auto lse_of = [&](uint32_t stats, int sub, int g) { l4[g & 1] = *(KR_LDS const f32x4*)(stats + 4 * (sub * 32 + 8 * g)); };
  auto s_mfma = [&](Scores& x, int kk) {
    if (kk == 0)
#pragma unroll
      for (int e = 0; e < 16; ++e) x.s[e] = 0.f;
    x.s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qfr[kk % 3], kf[kk], x.s, 0, 0, 0);
  };
  auto dp_mfma = [&](Scores& x, int kk) {
    x.dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dofr[kk % 3], vf[kk], x.dp, 0, 0, 0);
  };
  auto mask = [&](Scores& x, int qs0) {  // queries qs0 .. + 31; only blocks that reach the diagonal pay for it
    if (qs0 < kw0 + 31) {
      const int lim = krow - qs0 - 4 * h;  // element offsets below it are queries before the key
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float v = 8 * (e >> 2) + (e & 3) < lim ? -INFINITY : x.s[e];
        asm volatile("" : "+v"(v));  // keeps this a branch: off the diagonal no mask code runs
        x.s[e] = v;
      }
    }
  };
  // The three steps of a score.  Each result passes through an (empty) volatile asm: left alone the compiler moves the
  // work of several slots behind the next branch, away from the MFMAs that should cover it.
  auto score_a = [&](const Scores& x, int i) {
    x_at = __builtin_fmaf(x.s[i], scale_log2, l4[(i >> 2) & 1][i & 3]);
    asm volatile("" : "+v"(x_at));
  };
  auto score_b = [&]() {
    p_at = __builtin_amdgcn_exp2f(x_at);
    asm volatile("" : "+v"(p_at));
  };
  auto pack = [&](float lo, float hi) {
    bf16x2 v;
    v[0] = (bf16)lo;
    v[1] = (bf16)hi;
    uint32_t w = __builtin_bit_cast(uint32_t, v);
    asm volatile("" : "+v"(w));
    return w;
  };
  auto score_c = [&](const Scores& x, int i) {
    float ds = p_at * x.dp[i];
    asm volatile("" : "+v"(ds));
    if (i & 1) {
      pb[i >> 3][(i >> 1) & 3] = pack(p_even, p_at);
      dsb[i >> 3][(i >> 1) & 3] = pack(ds_even, ds);
    } else {
      p_even = p_at;
      ds_even = ds;
    }
  };
  // transposed fragment f of 16-query group k2: 2 dt: dO^T, 2 dt + 1: Q^T of channel block dt
  auto col_frag = [&](uint32_t cols, int sub, int k2, int f) {
    fr[f] = bt_cols<D>((f & 1) ? cols : cols + BT_BYTES, 2 * sub + k2, f >> 1);
  };
  // Block `sub` at (cols, stats); the block after it is n1 at (rows1, stats1), the one after that n2 at (rows2, stats2).
  auto block = [&](Scores& cur, Scores& nxt, uint32_t cols, uint32_t stats, int sub, uint32_t rows1, uint32_t stats1,
                   int n1, uint32_t rows2, uint32_t stats2, int n2, int qs1, auto&& behind_mfma, auto&& between) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (i == 10) {
        between();
        mask(nxt, qs1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (i < 8) {
        if (i & 1) dp_mfma(nxt, i >> 1);
        else s_mfma(nxt, i >> 1);
      } else {
        const int f = i & 3, k2 = (i - 8) >> 2, dt = f >> 1;
        const bf16x8 p8 = __builtin_bit_cast(bf16x8, (f & 1) ? dsb[k2] : pb[k2]);
        if (f & 1) dkacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[f], p8, dkacc[dt], 0, 0, 0);
        else dvacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[f], p8, dvacc[dt], 0, 0, 0);
      }
      behind_mfma(i);
      if (i == 0) row_frag(rows1, n1, 2);
      if (i == 2) row_frag(rows1, n1, 3);
      if (i >= 4 && i < 8) col_frag(cols, sub, 0, i - 4);
      if (i >= 8 && i < 12) col_frag(cols, sub, 1, i - 8);
      if (i == 2) lse_of(stats, sub, 3);
      if (i == 6 || i == 10 || i == 14) lse_of(stats1, n1, (i - 6) / 4);
      if (i < 12) score_c(cur, i + 4);
      else score_c(nxt, i - 12);
      score_b();
      if (i < 10) score_a(cur, i + 6);
      else score_a(nxt, i - 10);
      if (i == 12) row_frag(rows2, n2, 0);
      if (i == 14) row_frag(rows2, n2, 1);
      if (i >= 12) begin_dp(cur, stats2, n2, i - 12);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  if (nit_all > 0) {
    auto stage_of = [&](int it) { return lds0 + (it & (NS - 1)) * STAGE; };
    for (int t = 0; t < NS - 1 && t < nit_all; ++t) {
#pragma unroll
      for (int i = 0; i < 5; ++i) request_piece(stage_of(t), i);
      requested();
    }
    if (nit_all >= NS - 1)
      __builtin_amdgcn_s_waitcnt(0x0f75);  // vmcnt(5): all but the newest tile
    else
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    int qt = kt + part;  // query tile at hand
    const int qt_next = niter > 1 ? qt + qsplit : qt;
    zero_tail(lds0, qt);
    if (nit_all > 1) zero_tail(stage_of(1), qt_next);
    kr_barrier();
    settle_scalar_loads();
    const int qoff = 64 * half;  // this wave's queries of a tile
    Scores a, b;
    {
      const uint32_t rows = lds0 + rows_half, stats = lds0 + stat_lane;
#pragma unroll
      for (int g = 0; g < 4; ++g) begin_dp(a, stats, 0, g);
      lse_of(stats, 0, 0);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        row_frag(rows, 0, kk);
        s_mfma(a, kk);
        dp_mfma(a, kk);
      }
      mask(a, qt * TQ + qoff);
      lse_of(stats, 0, 1);
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        if (i >= 2) score_c(a, i - 2);
        if (i >= 1) score_b();
        score_a(a, i);
      }
      lse_of(stats, 0, 2);
      row_frag(rows, 1, 0);
      row_frag(rows, 1, 1);
#pragma unroll
      for (int g = 0; g < 4; ++g) begin_dp(b, stats, 1, g);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int it = 0; it < nit_all; ++it) {
      const uint32_t here = stage_of(it), there = stage_of(it + 1);
      uint32_t rows = here + rows_half, cols = here + cols_lane, stats = here + stat_lane;
      uint32_t rows_n = there + rows_half, stats_n = there + stat_lane;
      asm volatile("" : "+v"(rows), "+v"(cols), "+v"(stats), "+v"(rows_n), "+v"(stats_n));
      const int q0 = qt * TQ + qoff;
      qt = qt + qsplit >= nkt ? kt + part : qt + qsplit;  // of the next tile
      // from the last slots of block 0 on the next tile is read (behind the last one a stale stage, unused)
      block(a, b, cols, stats, 0, rows, stats, 1, rows_n, stats_n, 0, q0 + 32, [](int) {}, [&] {
        __builtin_amdgcn_s_waitcnt(0x0f75);  // vmcnt(5): of this wave's requests only those of tile it + 2 may be on their way
        if (it > 0 && it + 1 < nit_all) zero_tail(there, qt);  // (tiles 0 and 1 were settled before the loop)
        kr_barrier();  // everyone's share of tile it + 1 has landed, and nobody reads tile it - 1 any more
      });
      const uint32_t free = stage_of(it + NS - 1);
      block(b, a, cols, stats, 1, rows_n, stats_n, 0, rows_n, stats_n, 1, qt * TQ + qoff,
            [&](int i) { if (i < 5) request_piece(free, i); }, [] {});
      requested();
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the requests behind the last tile
  // The stages are free.  Wave w of the first half gives its dV to wave w of the second and gets its dK ([value][wave]
  // [lane] layout, 32 KB each); the first half stores dK, the second dV, through 4 KB per wave behind them.
  kr_barrier();
  float* xch = reinterpret_cast<float*>(smem) + wave * 64 + lane;
  float* mine = xch + half * (32 * 256);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) mine[(dt * 16 + e) * 256] = half == 0 ? dvacc[dt][e] : dkacc[dt][e];
  kr_barrier();
  const float* other = xch + (1 - half) * (32 * 256);
  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[dt][e] = (half == 0 ? dkacc[dt][e] : dvacc[dt][e]) + other[(dt * 16 + e) * 256];
  RowStage rs;
  rs.init(reinterpret_cast<char*>(smem) + 65536 + wave8 * 4096, lane);
  const float mul = half == 0 ? scale : 1.0f;
  if (PARTIAL) {
    const int64_t prow = (((int64_t)bi * nhg + hgroup) * qsplit + part) * sp + kw0;
    store_rows_f32<D>(rs, acc, mul, (half == 0 ? part_k : part_v) + prow * D, D);
  } else if (half == 0) {
    store_rows_bf16<D, RAGGED>(rs, acc, mul, dk + dkl.at(bi, kvh) + (int64_t)kw0 * dkl.s_, dkl.s_, s - kw0);
  } else {
    store_rows_bf16<D, RAGGED>(rs, acc, mul, dv + dvl.at(bi, kvh) + (int64_t)kw0 * dvl.s_, dvl.s_, s - kw0);
  }
}

// dk/dv[b, kvh, i, :] = sum over the group's query heads of the fp32 partials; one thread per
// 8 channels (two 16-byte reads per partial, one 16-byte bf16 store).
template <int D>
__global__ __launch_bounds__(256) void attn_group_reduce_kernel(
    const float* __restrict__ part_k, const float* __restrict__ part_v, bf16* __restrict__ dk,
    bf16* __restrict__ dv, int s, int sp, int nslots, int nkv, int qsplit, int64_t total, KLayout dkl, KLayout dvl) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (bi, kvh, si, chunk of 8)
  if (idx >= total) return;
  constexpr int VEC = D / 8;
  const int c = (int)(idx % VEC);
  const int si = (int)((idx / VEC) % s);
  const int kvh = (int)((idx / VEC) / s % nkv);
  const int bi = (int)((idx / VEC) / ((int64_t)s * nkv));
  const int per = nslots / nkv;  // partial results per KV head: one per workgroup that served the group
  float ak[8], av[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) ak[e] = av[e] = 0.f;
  for (int j = 0; j < per * qsplit; ++j) {  // (heads' workgroup, query-tile part) pairs are consecutive
    const int64_t off = (((((int64_t)bi * nslots + kvh * per) * qsplit + j) * sp) + si) * D + c * 8;
    const f32x4 k0 = *reinterpret_cast<const f32x4*>(part_k + off);
    const f32x4 k1 = *reinterpret_cast<const f32x4*>(part_k + off + 4);
    const f32x4 v0 = *reinterpret_cast<const f32x4*>(part_v + off);
    const f32x4 v1 = *reinterpret_cast<const f32x4*>(part_v + off + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      ak[e] += k0[e];
      ak[4 + e] += k1[e];
      av[e] += v0[e];
      av[4 + e] += v1[e];
    }
  }
  bf16x8 ok, ov;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    ok[e] = (bf16)ak[e];
    ov[e] = (bf16)av[e];
  }
  stg8(dk + dkl.at(bi, kvh) + (int64_t)si * dkl.s_ + c * 8, ok);
  stg8(dv + dvl.at(bi, kvh) + (int64_t)si * dvl.s_ + c * 8, ov);
}

// HALVES = 2: as in the forward kernel, two halves of an 8-wave workgroup own the same 128
// queries and walk the even / odd key tiles; half 1's dQ partial is added to half 0's through
// LDS at the end.  Chosen by the host when there are few workgroups.
// When there are more 256-query tiles than compute units (or other streams run beside the launch; see attn_forms)
// the host takes attn_bwd_dq_w64_kernel below instead.
template <int D, bool RAGGED, int HALVES>
__global__ __launch_bounds__(256 * HALVES, HALVES == 1 ? 2 : 1) void attn_bwd_dq_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    const bf16* __restrict__ dout, const float* __restrict__ lse, const float* __restrict__ neg_delta,
    bf16* __restrict__ dq, int s, int nq, int nkv, float scale, float scale_log2, QLayout ql,
    KLayout kl, KLayout vl, QLayout dol, QLayout dql) {
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];
  constexpr uint32_t STAGE = 2 * BT_BYTES;  // K tile | V tile (blocked tiles), bytes
  constexpr int TK = tile_rows<D>, NB = TK / 32, DT = D / 32, KK = D / 16;

  const int half = HALVES == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
  const int tid = threadIdx.x & 255, lane = tid & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int ROWS = BQ;  // queries per workgroup
  const int sp = RAGGED ? (s + 127) / 128 * 128 : s;
  const int nqt = sp / ROWS;
  int rank, pair;
  longest_first(blockIdx.x, gridDim.x, nqt, rank, pair);
  const int qt = nqt - 1 - rank;
  const int head = pair % nq;
  const int bi = pair / nq;
  const int per = nq / nkv;
  const int kvh = head / per;
  const int q0 = qt * ROWS;
  const int qw0 = q0 + wave * 32;
  const int qrow = qw0 + (lane & 31);
  const int qld = RAGGED && qrow >= s ? s - 1 : qrow;  // the row to load (rows beyond s are not stored)

  const bf16* qp = q + ql.at(bi, head, per) + (int64_t)qld * ql.s_;
  const bf16* dop = dout + dol.at(bi, head, per) + (int64_t)qld * dol.s_;
  const bf16* kb = k + kl.at(bi, kvh);
  const bf16* vb = v + vl.at(bi, kvh);
  bf16x8 qf[KK], dof[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    qf[kk] = ldg8(qp + kk * 16 + h * 8);
    dof[kk] = ldg8(dop + kk * 16 + h * 8);
  }
  const int64_t stat = (int64_t)bi * nq + head;
  const float neg_lse = -lse[stat * s + qld] * kLog2e;
  const float my_neg_delta = neg_delta[stat * sp + qld];

  f32x16 dqacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) dqacc[dt][e] = 0.f;

  // key tiles per half, up to the workgroup's last row (with 128-key tiles half 1 may have one less: its
  // last step then neither requests nor computes)
  const int ntiles = ((q0 + BQ) / TK + HALVES - 1) / HALVES;
  auto key_of = [&](int j) { return (HALVES * j + half) * TK; };
  // K and V tiles go straight from global memory into two LDS stages: this half's own, or with
  // shared tiles the workgroup's, half 0 bringing in the K tile and half 1 the V tile
  const uint32_t area = (uint32_t)(uintptr_t)(KR_LDS const bf16*)smem + half * 2 * STAGE;
  auto stage_request = [&](int j, int buf) {
    const int key0 = key_of(j);
    if (D == 64 && HALVES == 2 && key0 >= q0 + BQ) return;
    if (RAGGED && key0 + TK > s) {
      bt_request_clamped<D>(kb, kl.s_, key0, s, area + buf * STAGE, wave, lane);
      bt_request_clamped<D>(vb, vl.s_, key0, s, area + buf * STAGE + BT_BYTES, wave, lane);
      return;
    }
    bt_request<D>(kb + (int64_t)key0 * kl.s_, kl.s_, area + buf * STAGE, wave, lane);
    bt_request<D>(vb + (int64_t)key0 * vl.s_, vl.s_, area + buf * STAGE + BT_BYTES, wave, lane);
  };
  auto zero_tail = [&](int j, int buf) {  // rows of tile j beyond the sequence, once it has landed
    if (RAGGED && key_of(j) + TK > s) {
      bt_zero_tail<D>(key_of(j), s, area + buf * STAGE, wave, lane);
      bt_zero_tail<D>(key_of(j), s, area + buf * STAGE + BT_BYTES, wave, lane);
    }
  };
  stage_request(0, 0);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  zero_tail(0, 0);
  kr_barrier();

  settle_scalar_loads();
  for (int j = 0; j < ntiles; ++j) {
    const int cur = j & 1;
    if (j + 1 < ntiles) stage_request(j + 1, cur ^ 1);
    const int key0 = key_of(j);
    if (key0 <= qw0 + 31) {
      // one base register per tile and read direction; everything else is an immediate
      uint32_t k_rows = area + cur * STAGE + bt_rows_lane(lane);
      uint32_t v_rows = k_rows + BT_BYTES;
      uint32_t k_cols = area + cur * STAGE + bt_cols_lane(lane);
      asm volatile("" : "+v"(k_rows), "+v"(v_rows), "+v"(k_cols));
      const bool need_mask = key0 + TK - 1 > qw0;  // wave-uniform: the tile on the diagonal
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        if (D == 64 && key0 + 32 * t > qw0 + 31) continue;  // wave-uniform: beyond the diagonal
        f32x16 sacc, dpacc;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          sacc[e] = 0.f;
          dpacc[e] = 0.f;
        }
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bt_rows<D>(k_rows, t, kk), qf[kk], sacc, 0, 0, 0);
          dpacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bt_rows<D>(v_rows, t, kk), dof[kk], dpacc, 0, 0, 0);
        }
        // lane: query row qrow, keys key0 + 32t + 8g + 4h + e
        bf16x8 dsb[2];
        if (need_mask) {
          // Off the diagonal no mask code must run.  Left alone the compiler turns the branch
          // into 16 unconditional selects; values that pass through an (empty) volatile asm can
          // only be produced where the asm executes, i.e. inside the branch.
          const int lim = qrow - key0 - t * 32 - 4 * h;
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            float v = 8 * (e >> 2) + (e & 3) > lim ? -INFINITY : sacc[e];
            asm volatile("" : "+v"(v));
            sacc[e] = v;
          }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[e], scale_log2, neg_lse));
          dsb[e >> 3][e & 7] = (bf16)(p * (dpacc[e] + my_neg_delta));
        }
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            dqacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bt_cols<D>(k_cols, 2 * t + k2, dt), dsb[k2],
                                                                dqacc[dt], 0, 0, 0);
          }
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's share of the next tiles has landed
    if (RAGGED && j + 1 < ntiles) zero_tail(j + 1, cur ^ 1);
    kr_barrier();
  }

  if (HALVES == 2) {  // half 1 -> LDS -> half 0 ([value][wave][lane]; the staging areas are free)
    float* xch = reinterpret_cast<float*>(smem);
    const int slot = wave * 64 + lane;
    if (half == 1) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) xch[(dt * 16 + e) * 256 + slot] = dqacc[dt][e];
    }
    kr_barrier();
    if (half == 1) return;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) dqacc[dt][e] += xch[(dt * 16 + e) * 256 + slot];
  }

  // output transposition through LDS (behind the 64 KiB hand-over buffer when there are two halves)
  RowStage rs;
  rs.init(reinterpret_cast<char*>(smem) + (HALVES == 2 ? 64 * 1024 : 0) + wave * 4096, lane);
  store_rows_bf16<D, RAGGED>(rs, dqacc, scale, dq + dql.at(bi, head, per) + (int64_t)qw0 * dql.s_, dql.s_, s - qw0);
}

// ---------------------------------------------------------------------------------------------
// dQ with ONE wave per SIMD.  A wave owns 64 query rows (two blocks of 32) and all 512 registers of
// its lanes, so that every K / V fragment it reads from LDS feeds two MFMAs — a wave cannot fetch a
// 1 KB fragment faster than an MFMA takes, which is what holds the two-waves-per-SIMD kernels at
// half of the matrix pipe.  With a single instruction stream per SIMD nothing else would fill the
// pipe while the wave does its vector work, so the loop is software-pipelined by hand: behind each of
// the 32 score MFMAs (S^T, dP^T) of the NEXT 32 keys sits the multiply-add, exponential, multiplication
// and rounding of one score per lane of THIS step (dP^T comes out of its MFMAs with delta already
// subtracted), then come this step's 16 dQ MFMAs.
//
// The score MFMAs are inline assembly because their register file has to be chosen: a kernel with more
// than 256 registers gets its MFMA results in the accumulation registers, and every score would
// then pass through a copy before a vector instruction can read it.  Written by hand they land in
// ordinary VGPRs (with most Q / dO fragments in the accumulation registers, which the MFMA reads
// directly); the dQ MFMAs are ordinary builtins and keep dQ in the accumulation registers.  The
// compiler does not see an MFMA in the assembly, so the waits it would insert between such an
// instruction and a reader of its result are provided by construction:
//   * a score accumulator is read by vector instructions one step after the MFMAs that wrote it,
//     with that step's 16 dQ MFMAs in between (before the loop: explicit s_nop);
//   * score accumulators start from the instruction's zero operand or from a tuple set up before the
//     loop, never from a fresh vector write, and a result that is not also the addend is an
//     early-clobber operand (the instruction writes while it still reads).
// tests/test_attention_asm.py checks the compiled kernel for any reader that comes too early.
// Fragments come from LDS through ordinary loads, whose waits the compiler does insert.
// ---------------------------------------------------------------------------------------------
struct DqScores {
  f32x16 s[2], dp[2];  // per 32-query block: S^T and dP^T of 32 keys
};

// c = a . b / c += a . b with c in VGPRs; b in the accumulation registers or in VGPRs.  A result that
// is not also the addend must not share registers with the operands (early clobber): the
// instruction writes while it still reads.
__device__ __forceinline__ void mfma_set_v(f32x16& c, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma_acc_v(f32x16& c, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma_set_vv(f32x16& c, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma_acc_vv(f32x16& c, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}

// c = a . b + c0 with c and c0 in VGPRs (c0 is kept)
__device__ __forceinline__ void mfma_from_v(f32x16& c, bf16x8 a, bf16x8 b, const f32x16& c0) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(c) : "v"(a), "a"(b), "v"(c0));
}
__device__ __forceinline__ void mfma_from_vv(f32x16& c, bf16x8 a, bf16x8 b, const f32x16& c0) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(c) : "v"(a), "v"(b), "v"(c0));
}

// MFMA m (0..3) of contraction step kk: S^T of block 0, block 1, dP^T of block 0, block 1.  dP^T
// starts from -delta of the lane's row (sixteen copies per block, set up once), which takes the
// subtraction out of every score's vector work.
template <int KK>
__device__ __forceinline__ void dq_score_mfma(DqScores& x, int kk, int m, bf16x8 kf, bf16x8 vf,
                                              const bf16x8 (&qf)[2][KK], const bf16x8 (&dof)[2][KK],
                                              const f32x16 (&neg_delta)[2]) {
  if (kk == 0) {
    if (m == 0) mfma_set_v(x.s[0], kf, qf[0][kk]);
    if (m == 1) mfma_set_v(x.s[1], kf, qf[1][kk]);
    if (m == 2) mfma_from_v(x.dp[0], vf, dof[0][kk], neg_delta[0]);
    if (m == 3) mfma_from_vv(x.dp[1], vf, dof[1][kk], neg_delta[1]);
  } else {
    if (m == 0) mfma_acc_v(x.s[0], kf, qf[0][kk]);
    if (m == 1) mfma_acc_v(x.s[1], kf, qf[1][kk]);
    if (m == 2) mfma_acc_v(x.dp[0], vf, dof[0][kk]);
    if (m == 3) mfma_acc_vv(x.dp[1], vf, dof[1][kk]);
  }
}

// One step (32 keys).  NEXT: issue the score MFMAs of the following 32 keys (fragments of sub-tile nt
// at nk_rows / nv_rows) into `nxt`.  MASK: the step is on the causal diagonal; lim[qb] is the last
// visible key of the lane's row, relative to the lane's first key of the step.
template <int D, bool NEXT, bool MASK>
__device__ __forceinline__ void dq_step(DqScores& nxt, const DqScores& cur, f32x16 (&dq)[2][D / 32],
                                        uint32_t nk_rows, uint32_t nv_rows, int nt, uint32_t k_cols, int t,
                                        const bf16x8 (&qf)[2][D / 16], const bf16x8 (&dof)[2][D / 16],
                                        float scale_log2, const float (&neg_lse)[2],
                                        const f32x16 (&neg_delta)[2], const int (&lim)[2]) {
  constexpr int KK = D / 16, DT = D / 32;
  bf16x8 dsb[2][2];
  auto one_score = [&](int g) {  // lane: query row of block g / 16, key 8 (e / 4) + e % 4 (+ 4 h) of the step
    const int qb = g >> 4, e = g & 15;
    float sv = cur.s[qb][e];
    if (MASK) sv = 8 * (e >> 2) + (e & 3) > lim[qb] ? -INFINITY : sv;
    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sv, scale_log2, neg_lse[qb]));
    dsb[qb][e >> 3][e & 7] = (bf16)(p * cur.dp[qb][e]);  // dP - delta comes out of the MFMAs
  };
  // Fragments are requested from LDS well ahead of the MFMA that takes them (two contraction steps
  // = eight MFMAs for the score products, three fragments = six MFMAs for dQ): one wave per SIMD has
  // nobody to cover an LDS round trip for it.
  constexpr int NKT = 2 * (DT);  // K^T fragments of the step: 2 contraction steps x D / 32 channel blocks
  auto kt_frag = [&](int i) { return bt_cols<D>(k_cols, 2 * t + i / (DT), i % (DT)); };
  bf16x8 kt[3];
  if (NEXT) {
    bf16x8 kf[3], vf[3];
    kf[0] = bt_rows<D>(nk_rows, nt, 0);
    vf[0] = bt_rows<D>(nv_rows, nt, 0);
    kf[1] = bt_rows<D>(nk_rows, nt, 1);
    vf[1] = bt_rows<D>(nv_rows, nt, 1);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (m == 0 && kk + 2 < KK) kf[(kk + 2) % 3] = bt_rows<D>(nk_rows, nt, kk + 2);
        if (m == 2 && kk + 2 < KK) vf[(kk + 2) % 3] = bt_rows<D>(nv_rows, nt, kk + 2);
        if (m == 1 && kk >= KK - 3) kt[kk - (KK - 3)] = kt_frag(kk - (KK - 3));
        dq_score_mfma<KK>(nxt, kk, m, kf[kk % 3], vf[kk % 3], qf, dof, neg_delta);
#pragma unroll
        for (int c = 0; c < 8 / KK; ++c) one_score((kk * 4 + m) * (8 / KK) + c);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 3; ++i) kt[i] = kt_frag(i);
#pragma unroll
    for (int g = 0; g < 32; ++g) one_score(g);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 3");
  }
#pragma unroll
  for (int i = 0; i < NKT; ++i) {
    const int k2 = i / (DT), dt = i % (DT);
    const bf16x8 frag = kt[i % 3];
    dq[0][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag, dsb[0][k2], dq[0][dt], 0, 0, 0);
    dq[1][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag, dsb[1][k2], dq[1][dt], 0, 0, 0);
    if (i + 3 < NKT) kt[i % 3] = kt_frag(i + 3);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The kernel also takes over the pre-pass of the backward: each wave forms delta = sum_d dO . O of its 64
// rows from the dO fragments it holds anyway, uses it, and writes it (and -lse in the log2 domain) for
// the dK/dV kernel, which the host launches behind this one.
template <int D, bool RAGGED>
__global__ __launch_bounds__(256, 1) void attn_bwd_dq_w64_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    const bf16* __restrict__ dout, const bf16* __restrict__ o, const float* __restrict__ lse,
    float* __restrict__ neg_delta_out, float* __restrict__ neg_lse2_out, bf16* __restrict__ dq, int s, int nq,
    int nkv, float scale, float scale_log2, QLayout ql, KLayout kl, KLayout vl, QLayout dol, QLayout ol,
    QLayout dql) {
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];
  constexpr int TK = tile_rows<D>, NSUB = TK / 32, DT = D / 32, KK = D / 16;
  constexpr uint32_t STAGE = 2 * BT_BYTES;  // K tile | V tile
  constexpr int ROWS = 256;                 // queries per workgroup: 64 per wave
  constexpr int NSTAGE = 3;                 // tiles in LDS: the one in use, the next, the one after

  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sp = RAGGED ? (s + 127) / 128 * 128 : s;  // rows of the statistics (whole 256-query tiles here)
  const int nqt = sp / ROWS;
  int rank, pair;
  longest_first(blockIdx.x, gridDim.x, nqt, rank, pair);
  const int qt = nqt - 1 - rank;
  const int head = pair % nq;
  const int bi = pair / nq;
  const int per = nq / nkv;
  const int kvh = head / per;
  const int q0 = qt * ROWS;
  const int qw0 = q0 + wave * 64;

  const bf16* kb = k + kl.at(bi, kvh);
  const bf16* vb = v + vl.at(bi, kvh);
  bf16x8 qf[2][KK], dof[2][KK];
  float neg_lse[2];
  f32x16 neg_delta[2];
  int lim[2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int qrow = qw0 + 32 * qb + (lane & 31);
    const int qld = RAGGED && qrow >= s ? s - 1 : qrow;  // the row to load
    const bf16* qp = q + ql.at(bi, head, per) + (int64_t)qld * ql.s_;
    const bf16* dop = dout + dol.at(bi, head, per) + (int64_t)qld * dol.s_;
    const bf16* op = o + ol.at(bi, head, per) + (int64_t)qld * ol.s_;
    // delta from a second read of the dO row: the fragments kept for the MFMAs must stay values that
    // only the MFMAs read, or the compiler keeps them in VGPRs and copies them into accumulation
    // registers in front of every MFMA
    const bf16* dop2 = dop;
    asm volatile("" : "+v"(dop2));
    float dsum = 0.f;  // this lane's half of the row (channels 16 kk + 8 h ..)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      qf[qb][kk] = ldg8(qp + kk * 16 + h * 8);
      dof[qb][kk] = ldg8(dop + kk * 16 + h * 8);
      const bf16x8 dov = ldg8(dop2 + kk * 16 + h * 8), of = ldg8(op + kk * 16 + h * 8);
#pragma unroll
      for (int e = 0; e < 8; ++e) dsum += (float)dov[e] * (float)of[e];
    }
    dsum += __shfl_xor(dsum, 32, KR_WAVE);
    const int64_t stat = ((int64_t)bi * nq + head) * sp + qrow;
    neg_lse[qb] = -lse[((int64_t)bi * nq + head) * s + qld] * kLog2e;
    if (RAGGED && qrow >= s) {  // rows the dK/dV kernel must not see
      dsum = 0.f;
      neg_lse[qb] = -kPadLse * kLog2e;
    }
    if (h == 0) {
      neg_delta_out[stat] = -dsum;
      neg_lse2_out[stat] = neg_lse[qb];
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) neg_delta[qb][e] = -dsum;
  }

  f32x16 dqacc[2][DT];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) dqacc[qb][dt][e] = 0.f;

  const int ntiles = (q0 + ROWS) / TK;                              // key tiles of the workgroup
  const int last = __builtin_amdgcn_readfirstlane(qw0 / TK);        // this wave's tile on the diagonal
  const uint32_t area = (uint32_t)(uintptr_t)(KR_LDS const bf16*)smem;
  auto stage_request = [&](int j, int buf) {  // the four waves bring in the K and the V tile together
    if (RAGGED && (j + 1) * TK > s) {
      bt_request_clamped<D>(kb, kl.s_, j * TK, s, area + buf * STAGE, wave, lane);
      bt_request_clamped<D>(vb, vl.s_, j * TK, s, area + buf * STAGE + BT_BYTES, wave, lane);
      return;
    }
    bt_request<D>(kb + (int64_t)(j * TK) * kl.s_, kl.s_, area + buf * STAGE, wave, lane);
    bt_request<D>(vb + (int64_t)(j * TK) * vl.s_, vl.s_, area + buf * STAGE + BT_BYTES, wave, lane);
  };
  auto zero_tail = [&](int j, int buf) {  // rows of tile j beyond the sequence, once it has landed
    if (RAGGED && (j + 1) * TK > s) {
      bt_zero_tail<D>(j * TK, s, area + buf * STAGE, wave, lane);
      bt_zero_tail<D>(j * TK, s, area + buf * STAGE + BT_BYTES, wave, lane);
    }
  };
  stage_request(0, 0);
  stage_request(1, 1);  // ntiles >= 2
  __builtin_amdgcn_s_waitcnt(0x0f78);  // vmcnt(8): everything but the second tile's requests has landed
  zero_tail(0, 0);
  kr_barrier();
  settle_scalar_loads();

  const uint32_t rows_lane = bt_rows_lane(lane), cols_lane = bt_cols_lane(lane);
  DqScores a, b;
  {  // scores of the first 32 keys (tile 0 is below every wave's diagonal or on it)
    const uint32_t k_rows = area + rows_lane, v_rows = k_rows + BT_BYTES;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const bf16x8 kf = bt_rows<D>(k_rows, 0, kk), vf = bt_rows<D>(v_rows, 0, kk);
#pragma unroll
      for (int m = 0; m < 4; ++m) dq_score_mfma<KK>(a, kk, m, kf, vf, qf, dof, neg_delta);
    }
    // the scores pass through the wait: no reader can be moved in front of it
    asm volatile("s_nop 15\n\ts_nop 15" : "+v"(a.s[0]), "+v"(a.s[1]), "+v"(a.dp[0]), "+v"(a.dp[1]));
  }
  // Every wave passes the same ntiles barriers and makes the same requests; what differs is how many
  // of the tiles it computes on (those up to its diagonal).  Three loops without branches inside
  // (a branch around a step would put copies of all accumulators at the merge): tiles below the
  // diagonal, the diagonal tile, the tiles only the waves further down still need.
  int buf = 0;  // stage of tile j
  auto arrive = [&](int j) {  // between the two steps of tile j
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's share of tile j + 1 has landed
    if (RAGGED && j + 1 < ntiles) zero_tail(j + 1, buf == NSTAGE - 1 ? 0 : buf + 1);
    kr_barrier();                     // ... and everyone's; nobody reads tile j - 1 any more
  };
  auto turn = [&](int j) {
    arrive(j);
    if (j + NSTAGE - 1 < ntiles) stage_request(j + NSTAGE - 1, buf == 0 ? NSTAGE - 1 : buf - 1);
  };
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) lim[qb] = 0;
  for (int j = 0; j < last; ++j) {
    const int buf_next = buf == NSTAGE - 1 ? 0 : buf + 1;
    uint32_t k_rows = area + buf * STAGE + rows_lane, v_rows = k_rows + BT_BYTES;
    uint32_t k_cols = area + buf * STAGE + cols_lane;
    uint32_t nk_rows = area + buf_next * STAGE + rows_lane, nv_rows = nk_rows + BT_BYTES;
    asm volatile("" : "+v"(k_rows), "+v"(v_rows), "+v"(k_cols), "+v"(nk_rows), "+v"(nv_rows));
#pragma unroll
    for (int t = 0; t < NSUB; t += 2) {
      dq_step<D, true, false>(b, a, dqacc, k_rows, v_rows, t + 1, k_cols, t, qf, dof, scale_log2, neg_lse, neg_delta, lim);
      if (t + 2 < NSUB) {
        dq_step<D, true, false>(a, b, dqacc, k_rows, v_rows, t + 2, k_cols, t + 1, qf, dof, scale_log2, neg_lse, neg_delta, lim);
      } else {
        turn(j);
        dq_step<D, true, false>(a, b, dqacc, nk_rows, nv_rows, 0, k_cols, t + 1, qf, dof, scale_log2, neg_lse, neg_delta, lim);
      }
    }
    buf = buf_next;
  }
  {  // the tile on the diagonal: lim = last visible key of the lane's row, counted from the lane's first
     // key of the step (D = 64: the wave's 64 rows meet one half of the 128 keys; steps beyond the
     // diagonal are masked rather than branched around)
    uint32_t k_rows = area + buf * STAGE + rows_lane, v_rows = k_rows + BT_BYTES;
    uint32_t k_cols = area + buf * STAGE + cols_lane;
    asm volatile("" : "+v"(k_rows), "+v"(v_rows), "+v"(k_cols));
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) lim[qb] = 32 * qb + (lane & 31) - 4 * h + (D == 64 ? qw0 - last * TK : 0);
    auto next_keys = [&]() {
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) lim[qb] -= 32;
    };
#pragma unroll
    for (int t = 0; t < NSUB; t += 2) {
      dq_step<D, true, true>(b, a, dqacc, k_rows, v_rows, t + 1, k_cols, t, qf, dof, scale_log2, neg_lse, neg_delta, lim);
      next_keys();
      if (t + 2 < NSUB) {
        dq_step<D, true, true>(a, b, dqacc, k_rows, v_rows, t + 2, k_cols, t + 1, qf, dof, scale_log2, neg_lse, neg_delta, lim);
        next_keys();
      } else {
        turn(last);
        dq_step<D, false, true>(a, b, dqacc, 0, 0, 0, k_cols, t + 1, qf, dof, scale_log2, neg_lse, neg_delta, lim);
      }
    }
    buf = buf == NSTAGE - 1 ? 0 : buf + 1;
  }
  for (int j = last + 1; j < ntiles; ++j) {
    turn(j);
    buf = buf == NSTAGE - 1 ? 0 : buf + 1;
  }

  RowStage rs;
  rs.init(reinterpret_cast<char*>(smem) + NSTAGE * STAGE + wave * 4096, lane);
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
    store_rows_bf16<D, RAGGED>(rs, dqacc[qb], scale, dq + dql.at(bi, head, per) + (int64_t)(qw0 + 32 * qb) * dql.s_,
                               dql.s_, s - (qw0 + 32 * qb));
}

// =============================================================================================
// General path: any sequence length, head dimensions that are a multiple of 8 up to 128.
// The kernels above are built for head dimensions 128 and 64.  With KR_ATTN_GENERAL_KERNELS, or in the forward without
// a workspace, any shape but hd = 128 with whole 128-row tiles runs through these plain fp32 kernels:
// same interface, same tensor layouts, same results to rounding, no MFMA — they exist so that such a
// shape is computed on the device at all, not to be fast.  A workgroup of 256 threads owns 32
// query rows (forward, dQ) or 32 keys (dK/dV) and walks 32-row tiles of the other operand through
// LDS; a thread is (row r = tid / 8, part p = tid % 8): it computes the scores of row r against
// keys 4 p .. 4 p + 3 of a tile and owns channels p hd/8 .. (p + 1) hd/8 - 1 of row r's
// accumulators.  Rows beyond the sequence are loaded as zeros and never stored.  No atomics:
// grouped query heads are summed inside the dK/dV workgroup, in a fixed order.
// =============================================================================================
namespace general {

constexpr int GT = 32;          // rows per tile (queries or keys)
constexpr int GTHREADS = 256;
constexpr int GHD_MAX = 128;
constexpr int GLD = GHD_MAX + 8;  // LDS row stride in elements (rows stay 16-byte aligned)

// rows row0 .. row0 + 31 of a [s, hd] matrix with row stride ss -> LDS tile, zeros beyond s
__device__ __forceinline__ void load_tile(bf16* dst, const bf16* src, int64_t ss, int row0, int s,
                                          int hd, int tid) {
  const int vecs = hd / 8;
  for (int i = tid; i < GT * vecs; i += GTHREADS) {
    const int r = i / vecs, c = (i - r * vecs) * 8;
    const bf16x8 v = row0 + r < s ? ldg8(src + (int64_t)(row0 + r) * ss + c) : zero8();
    *reinterpret_cast<bf16x8*>(dst + r * GLD + c) = v;
  }
}

// sum / max over the 8 threads that share a row (consecutive lanes)
__device__ __forceinline__ float row_sum(float v) {
  v += __shfl_xor(v, 1, KR_WAVE);
  v += __shfl_xor(v, 2, KR_WAVE);
  v += __shfl_xor(v, 4, KR_WAVE);
  return v;
}
__device__ __forceinline__ float row_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 1, KR_WAVE));
  v = fmaxf(v, __shfl_xor(v, 2, KR_WAVE));
  v = fmaxf(v, __shfl_xor(v, 4, KR_WAVE));
  return v;
}

// dot products of row `r` of tile a with rows 4 p .. 4 p + 3 of tile b over hd channels
__device__ __forceinline__ void dot4(const bf16* a, const bf16* b, int r, int p, int hd, float (&out)[4]) {
  out[0] = out[1] = out[2] = out[3] = 0.f;
  const bf16* ar = a + r * GLD;
  const bf16* b0 = b + (4 * p) * GLD;
  for (int d = 0; d < hd; ++d) {
    const float av = (float)ar[d];
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] += av * (float)b0[j * GLD + d];
  }
}

__global__ __launch_bounds__(GTHREADS) void attn_general_fwd_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    bf16* __restrict__ o, float* __restrict__ lse, int s, int nq, int nkv, int hd, float scale,
    QLayout ql, KLayout kl, KLayout vl, QLayout ol) {
  __shared__ __attribute__((aligned(16))) bf16 sq[GT * GLD], sk[GT * GLD], sv[GT * GLD];
  __shared__ float sp[GT][GT + 1];
  const int tid = threadIdx.x, r = tid >> 3, p = tid & 7;
  const int q0 = blockIdx.x * GT, head = blockIdx.y, bi = blockIdx.z;
  const int per = nq / nkv, kvh = head / per, c = hd / 8;
  const bf16* qb = q + ql.at(bi, head, per);
  const bf16* kb = k + kl.at(bi, kvh);
  const bf16* vb = v + vl.at(bi, kvh);
  load_tile(sq, qb, ql.s_, q0, s, hd, tid);
  float acc[GHD_MAX / 8];
#pragma unroll
  for (int i = 0; i < GHD_MAX / 8; ++i) acc[i] = 0.f;
  float m = -INFINITY, l = 0.f;
  const int qrow = q0 + r;
  const int last_key = (q0 + GT - 1 < s ? q0 + GT - 1 : s - 1);
  for (int k0 = 0; k0 <= last_key; k0 += GT) {
    kr_barrier();  // the previous tile's K, V and probabilities are no longer read
    load_tile(sk, kb, kl.s_, k0, s, hd, tid);
    load_tile(sv, vb, vl.s_, k0, s, hd, tid);
    kr_barrier();
    float sc[4];
    dot4(sq, sk, r, p, hd, sc);
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int key = k0 + 4 * p + j;
      sc[j] = (key <= qrow && key < s) ? sc[j] * scale : -INFINITY;
      mx = fmaxf(mx, sc[j]);
    }
    mx = row_max(mx);
    const float m_new = fmaxf(m, mx);
    float pr[4], ps = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      pr[j] = sc[j] == -INFINITY ? 0.f : __expf(sc[j] - m_new);
      ps += pr[j];
      sp[r][4 * p + j] = pr[j];
    }
    ps = row_sum(ps);
    const float alpha = m == -INFINITY ? 0.f : __expf(m - m_new);
    l = l * alpha + ps;
    m = m_new;
    kr_barrier();
    for (int i = 0; i < c; ++i) acc[i] *= alpha;
    for (int kj = 0; kj < GT; ++kj) {
      const float pv = sp[r][kj];
      const bf16* vr = sv + kj * GLD + p * c;
      for (int i = 0; i < c; ++i) acc[i] += pv * (float)vr[i];
    }
  }
  if (qrow < s) {
    const float inv = 1.0f / l;
    bf16* orow = o + ol.at(bi, head, per) + (int64_t)qrow * ol.s_ + p * c;
    for (int i = 0; i < c; ++i) orow[i] = (bf16)(acc[i] * inv);
    if (p == 0) lse[((int64_t)bi * nq + head) * s + qrow] = m + __logf(l);
  }
}

// delta[b, h, i] = sum_d dO[i, d] O[i, d]
__global__ __launch_bounds__(GTHREADS) void attn_general_delta_kernel(
    const bf16* __restrict__ dout, const bf16* __restrict__ o, float* __restrict__ delta, int s,
    int nq, int nkv, int hd, QLayout dol, QLayout ol) {
  const int tid = threadIdx.x, r = tid >> 3, p = tid & 7;
  const int row = blockIdx.x * GT + r, head = blockIdx.y, bi = blockIdx.z;
  const int per = nq / nkv, c = hd / 8;
  float sum = 0.f;
  if (row < s) {
    const bf16* dr = dout + dol.at(bi, head, per) + (int64_t)row * dol.s_ + p * c;
    const bf16* orow = o + ol.at(bi, head, per) + (int64_t)row * ol.s_ + p * c;
    for (int i = 0; i < c; ++i) sum += (float)dr[i] * (float)orow[i];
  }
  sum = row_sum(sum);
  if (row < s && p == 0) delta[((int64_t)bi * nq + head) * s + row] = sum;
}

// P and dS of one 32 x 32 block: thread (r, p) handles query row r against keys 4 p .. 4 p + 3
__device__ __forceinline__ void block_p_ds(const bf16* sq, const bf16* sk, const bf16* sv, const bf16* sdo,
                                           const float* slse, const float* sdelta, int r, int p, int hd,
                                           int q0, int k0, int s, float scale, float (&pr)[4],
                                           float (&ds)[4]) {
  float sc[4], dp[4];
  dot4(sq, sk, r, p, hd, sc);
  dot4(sdo, sv, r, p, hd, dp);
  const int qrow = q0 + r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int key = k0 + 4 * p + j;
    const bool valid = key <= qrow && key < s && qrow < s;
    pr[j] = valid ? __expf(sc[j] * scale - slse[r]) : 0.f;
    ds[j] = pr[j] * (dp[j] - sdelta[r]) * scale;
  }
}

__global__ __launch_bounds__(GTHREADS) void attn_general_dkdv_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    const bf16* __restrict__ dout, const float* __restrict__ lse, const float* __restrict__ delta,
    bf16* __restrict__ dk, bf16* __restrict__ dv, int s, int nq, int nkv, int hd, float scale,
    QLayout ql, KLayout kl, KLayout vl, QLayout dol, KLayout dkl, KLayout dvl) {
  __shared__ __attribute__((aligned(16))) bf16 sq[GT * GLD], sk[GT * GLD], sv[GT * GLD], sdo[GT * GLD];
  __shared__ float sp[GT][GT + 1], sds[GT][GT + 1], slse[GT], sdelta[GT];
  const int tid = threadIdx.x, r = tid >> 3, p = tid & 7;
  const int k0 = blockIdx.x * GT, kvh = blockIdx.y, bi = blockIdx.z;
  const int per = nq / nkv, c = hd / 8;
  load_tile(sk, k + kl.at(bi, kvh), kl.s_, k0, s, hd, tid);
  load_tile(sv, v + vl.at(bi, kvh), vl.s_, k0, s, hd, tid);
  float adk[GHD_MAX / 8], adv[GHD_MAX / 8];
#pragma unroll
  for (int i = 0; i < GHD_MAX / 8; ++i) adk[i] = adv[i] = 0.f;
  for (int hj = 0; hj < per; ++hj) {
    const int head = kvh * per + hj;
    const bf16* qb = q + ql.at(bi, head, per);
    const bf16* dob = dout + dol.at(bi, head, per);
    const int64_t stat = ((int64_t)bi * nq + head) * s;
    for (int q0 = k0; q0 < s; q0 += GT) {  // query tiles at or below the diagonal (k0 is a multiple of 32)
      kr_barrier();
      load_tile(sq, qb, ql.s_, q0, s, hd, tid);
      load_tile(sdo, dob, dol.s_, q0, s, hd, tid);
      if (tid < GT) {
        const bool in = q0 + tid < s;
        slse[tid] = in ? lse[stat + q0 + tid] : 0.f;
        sdelta[tid] = in ? delta[stat + q0 + tid] : 0.f;
      }
      kr_barrier();
      float pr[4], ds[4];
      block_p_ds(sq, sk, sv, sdo, slse, sdelta, r, p, hd, q0, k0, s, scale, pr, ds);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sp[r][4 * p + j] = pr[j];
        sds[r][4 * p + j] = ds[j];
      }
      kr_barrier();
      // this thread now is (key r, channels p c ..): dV += P^T dO, dK += dS^T Q
      for (int qi = 0; qi < GT; ++qi) {
        const float pv = sp[qi][r], dsv = sds[qi][r];
        const bf16* dor = sdo + qi * GLD + p * c;
        const bf16* qr = sq + qi * GLD + p * c;
        for (int i = 0; i < c; ++i) {
          adv[i] += pv * (float)dor[i];
          adk[i] += dsv * (float)qr[i];
        }
      }
    }
  }
  if (k0 + r < s) {
    bf16* dkr = dk + dkl.at(bi, kvh) + (int64_t)(k0 + r) * dkl.s_ + p * c;
    bf16* dvr = dv + dvl.at(bi, kvh) + (int64_t)(k0 + r) * dvl.s_ + p * c;
    for (int i = 0; i < c; ++i) {
      dkr[i] = (bf16)adk[i];
      dvr[i] = (bf16)adv[i];
    }
  }
}

__global__ __launch_bounds__(GTHREADS) void attn_general_dq_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    const bf16* __restrict__ dout, const float* __restrict__ lse, const float* __restrict__ delta,
    bf16* __restrict__ dq, int s, int nq, int nkv, int hd, float scale, QLayout ql, KLayout kl,
    KLayout vl, QLayout dol, QLayout dql) {
  __shared__ __attribute__((aligned(16))) bf16 sq[GT * GLD], sk[GT * GLD], sv[GT * GLD], sdo[GT * GLD];
  __shared__ float sds[GT][GT + 1], slse[GT], sdelta[GT];
  const int tid = threadIdx.x, r = tid >> 3, p = tid & 7;
  const int q0 = blockIdx.x * GT, head = blockIdx.y, bi = blockIdx.z;
  const int per = nq / nkv, kvh = head / per, c = hd / 8;
  const int64_t stat = ((int64_t)bi * nq + head) * s;
  load_tile(sq, q + ql.at(bi, head, per), ql.s_, q0, s, hd, tid);
  load_tile(sdo, dout + dol.at(bi, head, per), dol.s_, q0, s, hd, tid);
  if (tid < GT) {
    const bool in = q0 + tid < s;
    slse[tid] = in ? lse[stat + q0 + tid] : 0.f;
    sdelta[tid] = in ? delta[stat + q0 + tid] : 0.f;
  }
  const bf16* kb = k + kl.at(bi, kvh);
  const bf16* vb = v + vl.at(bi, kvh);
  float adq[GHD_MAX / 8];
#pragma unroll
  for (int i = 0; i < GHD_MAX / 8; ++i) adq[i] = 0.f;
  const int last_key = (q0 + GT - 1 < s ? q0 + GT - 1 : s - 1);
  for (int k0 = 0; k0 <= last_key; k0 += GT) {
    kr_barrier();
    load_tile(sk, kb, kl.s_, k0, s, hd, tid);
    load_tile(sv, vb, vl.s_, k0, s, hd, tid);
    kr_barrier();
    float pr[4], ds[4];
    block_p_ds(sq, sk, sv, sdo, slse, sdelta, r, p, hd, q0, k0, s, scale, pr, ds);
#pragma unroll
    for (int j = 0; j < 4; ++j) sds[r][4 * p + j] = ds[j];
    kr_barrier();
    for (int kj = 0; kj < GT; ++kj) {
      const float dsv = sds[r][kj];
      const bf16* kr = sk + kj * GLD + p * c;
      for (int i = 0; i < c; ++i) adq[i] += dsv * (float)kr[i];
    }
  }
  if (q0 + r < s) {
    bf16* dqr = dq + dql.at(bi, head, per) + (int64_t)(q0 + r) * dql.s_ + p * c;
    for (int i = 0; i < c; ++i) dqr[i] = (bf16)adq[i];
  }
}

}  // namespace general

// ---- shapes outside the MFMA kernels, padded into them -----------------------------------------
// Head dimensions other than 128 and 64 (and strides that attn_in_place refuses) are copied into
// dense [s_pad, b, heads, 128] buffers (zeros beyond the data), run through the MFMA kernels and
// copied back.  Zero channels add nothing to Q.K^T and give zero output channels; with the causal
// mask a query row below s never sees a key row at or beyond s, and the rows at or beyond s are
// made inert in the backward pass by a log-sum-exp so large that their probabilities are zero.
__global__ __launch_bounds__(256) void attn_pad_kernel(const bf16* __restrict__ src, bf16* __restrict__ dst,
                                                       int s, int b, int heads, int per, int hd,
                                                       int64_t total, QLayout sl) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one 16-byte vector of dst
  if (idx >= total) return;
  const int c = (int)(idx & 15) * 8;
  int64_t r = idx >> 4;
  const int head = (int)(r % heads);
  r /= heads;
  const int bi = (int)(r % b);
  const int row = (int)(r / b);
  bf16x8 v = zero8();
  if (row < s && c < hd) v = ldg8(src + (int64_t)row * sl.s_ + sl.at(bi, head, per) + c);
  stg8(dst + idx * 8, v);
}
__global__ __launch_bounds__(256) void attn_unpad_kernel(const bf16* __restrict__ src, bf16* __restrict__ dst,
                                                         int b, int heads, int per, int hd,
                                                         int64_t total, QLayout dl) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one 16-byte vector of dst
  if (idx >= total) return;
  const int vec = hd / 8;
  const int c = (int)(idx % vec) * 8;
  int64_t r = idx / vec;
  const int head = (int)(r % heads);
  r /= heads;
  const int bi = (int)(r % b);
  const int64_t row = r / b;
  const bf16x8 v = ldg8(src + (((row * b + bi) * heads + head) * HD + c));
  stg8(dst + row * dl.s_ + dl.at(bi, head, per) + c, v);
}
// rows of fp32 statistics [n, len_src] -> [n, len_dst]; positions beyond len_src get `fill`
__global__ __launch_bounds__(256) void attn_resize_rows_kernel(const float* __restrict__ src,
                                                               float* __restrict__ dst, int len_src,
                                                               int len_dst, int64_t total, float fill) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= total) return;
  const int64_t row = idx / len_dst;
  const int i = (int)(idx - row * len_dst);
  dst[idx] = i < len_src ? src[row * len_src + i] : fill;
}

}  // namespace

// Build-time cap, for measuring one form of a kernel against another: the most query heads a
// dK/dV workgroup takes.
#ifndef KR_DKDV_HPW_MAX
#define KR_DKDV_HPW_MAX 4
#endif
// The dK/dV kernels run one workgroup per CU.  With few of them their time is set by the first key tiles (they see every
// query): two workgroups then share each key tile, which costs fp32 partial sums and a launch that adds them.  At head
// dimension 64 the halves of a workgroup share a key tile's queries already, so that pays only for long rows and, where the heads
// of a group leave partial sums anyway, for few workgroups (whole -> split, with the launch that adds, us): 8 heads at s 200, b 2
// 10.2 -> 13.5, at s 1000 19.3 -> 18.9, at s 1000, b 4 21.8 -> 33.7; at s 1536 23.1 -> 24.9; one head at s 4096 47.0 -> 32.6, 4 heads
// 50.2 -> 38.4; in groups 6 heads at s 3072 45.6 -> 34.7, 8 heads at s 1024 23.0 -> 20.8, s 512 16.9 -> 16.0, s 256 13.8 -> 13.6, 16 heads
// 17.8 -> 18.2 and 14.2 -> 14.6 at the last two, one tile 12.3 -> 12.8.
// At head dimension 128, by the number of (key tile, head) pairs against the units (us with the launch that adds; whole and split,
// 2h: with two heads of a group to a workgroup).  Fewer pairs than units: split (64 64, 44; 128 119, 88; 192 at s 1504 63, 45),
// but not short rows that leave few units idle (192 at s 512 28, 32; in groups, by key tiles: 4 144 28, 26, 160 28, 29; 5 160 31.4, 29.9,
// 180 32.4, 33.4; 6 168 34.6, 33.0, 192 35.5, 34.9, 240 37.8, 41.7; 7 168 38.0, 33.8, 224 40.4, 40.6; without groups whole stores no
// partial sums: 5 160 24.1, 30.3, 6 168 28.0, 34.3, 7 168 31.5, 34.3).  One each: long rows (s 2048 69, 60; s 1024 45, 49).  More:
// whole (384 at s 2048 81 and 92, 102 and 113; at s 4096 149, 160; 480 at s 2048 97, 116; 496 at s 3968 156, 175).  Two each is the
// one count that has room for two parts (below) and leaves two workgroups a unit when each takes two heads: 2h (s 512 52.6, 51.4;
// s 1024 65.4, 64.1; s 2048 98.5, 97.1; s 4096 164.8, 163.3), where the XCDs get equal shares of it (4 head groups at s 8192 301, 403).
static int dkdv_query_split(int s, int b, int nq, int nkv, int hd) {
  const int key_tiles = s / 128, pairs = key_tiles * nq * b, cus = kr_compute_units();
  if (hd == 64) return (2 * pairs <= cus && key_tiles >= 16) || (nq != nkv && key_tiles >= 2 && pairs <= 8 * key_tiles && pairs <= cus) ? 2 : 1;
  if (pairs < cus) return 2 * pairs <= cus || (nq != nkv ? 8 * pairs <= cus * key_tiles : key_tiles >= 8) ? 2 : 1;
  if (4 * pairs < 5 * cus) return key_tiles >= 16 ? 2 : 1;
  return pairs == 2 * cus && (nq / nkv) % 2 == 0 && (nq / 2 * b) % kXcds == 0 ? 2 : 1;
}
// how many the workspace has room for
static int dkdv_query_split_reserved(int s, int b, int nq) { return (s / 128) * nq * b <= 2 * 256 ? 2 : 1; }

static int attn_padded_len(int s) { return (s + BQ - 1) / BQ * BQ; }
// bytes of one padded [s_pad, b, heads, 128] bf16 tensor / of the padded statistics [b, nq, s_pad]
static size_t attn_padded_bytes(int s, int b, int heads) {
  return (size_t)attn_padded_len(s) * b * heads * HD * sizeof(bf16);
}
static size_t attn_padded_stat_bytes(int s, int b, int nq) {
  return (size_t)attn_padded_len(s) * b * nq * sizeof(float);
}

// workspace of the MFMA backward kernels for a shape they take as it is
static size_t attn_bwd_fast_bytes(int s, int b, int nq, int nkv, int hd) {
  size_t bytes = 2 * (size_t)b * nq * s * sizeof(float);  // delta, and -lse in the log2 domain
  const int qsplit = dkdv_query_split_reserved(s, b, nq);
  if (nq != nkv || qsplit > 1)  // fp32 dK, dV partials per (query head, query-tile part)
    bytes += 2 * (size_t)b * nq * qsplit * s * hd * sizeof(float);
  return bytes;
}

extern "C" size_t kr_attn_bwd_workspace_bytes(int s, int b, int nq, int nkv, int hd) {
  if (check_attn_common(s, b, nq, nkv, hd) != KR_OK) return 0;
  if (attn_fast_path(s, hd)) return attn_bwd_fast_bytes(s, b, nq, nkv, hd);
  // padded copies of dO, q, o, dq (query-sized) and k, v, dk, dv (key-sized), the padded log-sum-exp, and
  // the MFMA kernels' own workspace at the padded shape (the general kernels, which only keep delta
  // [b, nq, s], fit in the same space)
  return 4 * attn_padded_bytes(s, b, nq) + 4 * attn_padded_bytes(s, b, nkv) + attn_padded_stat_bytes(s, b, nq) +
         attn_bwd_fast_bytes(attn_padded_len(s), b, nq, nkv, HD);
}

extern "C" size_t kr_attn_fwd_workspace_bytes(int s, int b, int nq, int nkv, int hd) {
  if (check_attn_common(s, b, nq, nkv, hd) != KR_OK || attn_fast_path(s, hd)) return 0;
  // padded copies of q, o and k, v, and the padded log-sum-exp
  return 2 * attn_padded_bytes(s, b, nq) + 2 * attn_padded_bytes(s, b, nkv) + attn_padded_stat_bytes(s, b, nq);
}

// The sizes above hold for any strides.  A caller who knows them need not reserve the copies of a shape that is
// not copied: s 4096, b 2, 32/8 heads of 64 asks for 169 MB forward and 607 MB backward above, for 0 and
// 136 MB (statistics and fp32 partial sums) here.
extern "C" size_t kr_attn_fwd_workspace_bytes_strided(int s, int b, int nq, int nkv, int hd, int64_t max_seq_stride) {
  return attn_in_place(s, hd, {max_seq_stride}) ? 0 : kr_attn_fwd_workspace_bytes(s, b, nq, nkv, hd);
}
extern "C" size_t kr_attn_bwd_workspace_bytes_strided(int s, int b, int nq, int nkv, int hd, int64_t max_seq_stride) {
  if (check_attn_common(s, b, nq, nkv, hd) != KR_OK) return 0;
  return attn_in_place(s, hd, {max_seq_stride}) ? attn_bwd_fast_bytes(attn_padded_len(s), b, nq, nkv, hd)
                                                : kr_attn_bwd_workspace_bytes(s, b, nq, nkv, hd);
}

namespace {
// dense [s_pad, b, heads, 128] as the kernels' stride quadruple / triple
QLayout padded_qlayout(int b, int nq, int per) {
  return QLayout{(int64_t)b * nq * HD, (int64_t)nq * HD, (int64_t)per * HD, (int64_t)HD};
}
KLayout padded_klayout(int b, int nkv) { return KLayout{(int64_t)b * nkv * HD, (int64_t)nkv * HD, (int64_t)HD}; }

int launch_pad(const void* src, void* dst, int s, int b, int heads, int per, int hd, QLayout sl, hipStream_t st) {
  const int64_t total = (int64_t)attn_padded_len(s) * b * heads * (HD / 8);
  hipLaunchKernelGGL(attn_pad_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, (const bf16*)src,
                     (bf16*)dst, s, b, heads, per, hd, total, sl);
  return hipGetLastError() == hipSuccess ? KR_OK : KR_ELAUNCH;
}
int launch_unpad(const void* src, void* dst, int s, int b, int heads, int per, int hd, QLayout dl, hipStream_t st) {
  const int64_t total = (int64_t)s * b * heads * (hd / 8);
  hipLaunchKernelGGL(attn_unpad_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, (const bf16*)src,
                     (bf16*)dst, b, heads, per, hd, total, dl);
  return hipGetLastError() == hipSuccess ? KR_OK : KR_ELAUNCH;
}
int launch_resize_rows(const float* src, float* dst, int64_t n, int len_src, int len_dst, float fill, hipStream_t st) {
  const int64_t total = n * len_dst;
  hipLaunchKernelGGL(attn_resize_rows_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, src, dst,
                     len_src, len_dst, total, fill);
  return hipGetLastError() == hipSuccess ? KR_OK : KR_ELAUNCH;
}
// a KV-like tensor's stride triple as the quadruple the pad kernels take (one head per group)
QLayout as_qlayout(const KLayout& l) { return QLayout{l.s_, l.b_, l.h_, 0}; }
}  // namespace

// Which form of each kernel a launch takes.  Alone on the GPU a launch wants the shortest latency:
// with few workgroups the keys of a row (forward, dQ) or the queries of a key tile (dK/dV) are split
// over two workgroups, which fills the device and costs merges, partial sums and a second pass over
// K / V.  Beside kernels of other streams (KR_ATTN_BESIDE_OTHER_STREAMS), which use the compute
// units a launch leaves idle, its compute-unit time counts instead: the unsplit forms, whatever the
// number of workgroups.
struct AttnForms {
  bool shared_fwd, shared_dq;
  int qsplit;
};
// One 256-query tile for every unit is not enough for the unsplit forms unless the rows are short: the longest row is then the
// launch (split forms -> unsplit, us: 8 pairs at s 8192 forward 134 -> 183, dQ 199 -> 247; 32 pairs at s 2048 47 -> 54, 68 -> 88;
// 64 at s 1024 30 -> 31, 44 -> 45; 128 at s 512 24 -> 20, 30 -> 32; at nine eighths of that, 32 pairs at s 2304, 67 -> 65, 104 -> 91).
static AttnForms attn_forms(int s, int b, int nq, int nkv, int hd, int flags) {  // s: rounded up to whole 128-row tiles
  const bool beside = (flags & KR_ATTN_BESIDE_OTHER_STREAMS) != 0;
  const int tiles256 = (s / 256) * nq * b, cus = kr_compute_units();
  const bool unsplit = s % 256 == 0 && (beside || tiles256 > cus || (tiles256 == cus && s <= 1024));
  AttnForms f;
  f.shared_fwd = f.shared_dq = unsplit;
  const int split = beside ? 1 : dkdv_query_split(s, b, nq, nkv, hd), room = dkdv_query_split_reserved(s, b, nq);
  f.qsplit = split < room ? split : room;
  return f;
}

namespace {
struct BwdCall {
  const bf16 *dout, *q, *k, *v, *o;
  const float* lse;
  bf16 *dq, *dk, *dv;
  float* workspace;
  int s, b, nq, nkv;
  float scale;
  QLayout ql, ol, dol, dql;
  KLayout kl, vl, dkl, dvl;
  int flags;
  hipStream_t st;
};

// The MFMA backward on tensors as they lie.  The forms are chosen by the length rounded up to whole 128-row
// tiles: the kernels walk those, whatever part of the last one exists.
template <int D, bool RAGGED>
int attn_bwd_mfma(const BwdCall& c) {
  const bf16 *dout = c.dout, *q = c.q, *k = c.k, *v = c.v, *o = c.o;
  const float* lse = c.lse;
  bf16 *dq = c.dq, *dk = c.dk, *dv = c.dv;
  const int s = c.s, b = c.b, nq = c.nq, nkv = c.nkv, sp = attn_padded_len(s);
  const float scale = c.scale;
  const QLayout ql = c.ql, ol = c.ol, dol = c.dol, dql = c.dql;
  const KLayout kl = c.kl, vl = c.vl, dkl = c.dkl, dvl = c.dvl;
  hipStream_t st = c.st;
  float* neg_delta = c.workspace;
  const int64_t rows = (int64_t)b * nq * sp;
  float* neg_lse2 = neg_delta + rows;
  float* part_k = neg_lse2 + rows;
  const AttnForms forms = attn_forms(sp, b, nq, c.nkv, D, c.flags);
  const int qsplit = forms.qsplit;
  float* part_v = part_k + rows * qsplit * D;
  // query heads of a KV group per dK/dV workgroup: as many as leave two workgroups per compute
  // unit (KR_DKDV_HPW_MAX: a build-time cap, for measurements)
  int hpw = 1;
  {
    const int per_group = nq / nkv;
    const int64_t wgs = (int64_t)(sp / 128) * nq * b * qsplit;
    for (int h2 = per_group < KR_DKDV_HPW_MAX ? per_group : KR_DKDV_HPW_MAX; h2 > 1; --h2)
      if (per_group % h2 == 0 && wgs / h2 >= 2 * (int64_t)kr_compute_units()) {
        hpw = h2;
        break;
      }
  }
  const bool partial = nq / hpw != nkv || qsplit > 1;
  // D = 128: three stages and the hand-over area; D = 64: four stages
  constexpr size_t lds_dkdv = D == 64 ? 4 * (2 * BT_BYTES + 8 * tile_rows<D>) : 3 * (2 * BT_BYTES + 8 * tile_rows<D>) + 32768;
  const auto dkdv_kernel = [](bool partial) {
    if constexpr (D == 64)
      return partial ? attn_bwd_dkdv64_kernel<RAGGED, true> : attn_bwd_dkdv64_kernel<RAGGED, false>;
    else
      return partial ? attn_bwd_dkdv_kernel<RAGGED, true> : attn_bwd_dkdv_kernel<RAGGED, false>;
  };
  constexpr size_t lds_dq = 2 * (2 * BT_BYTES);  // two stages of a K and a V tile
  constexpr size_t lds_dq_w64 = 3 * (2 * BT_BYTES) + 4 * 4096;  // three stages + a 4 KB output stage per wave
  static const hipError_t attr_status = [&] {
    hipError_t e = hipFuncSetAttribute((const void*)dkdv_kernel(false), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds_dkdv);
    if (e == hipSuccess)
      e = hipFuncSetAttribute((const void*)dkdv_kernel(true), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_dkdv);
    if (e == hipSuccess)
      e = hipFuncSetAttribute((const void*)attn_bwd_dq_kernel<D, RAGGED, 1>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_dq);
    if (e == hipSuccess)
      e = hipFuncSetAttribute((const void*)attn_bwd_dq_kernel<D, RAGGED, 2>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)(2 * lds_dq));
    if (e == hipSuccess)
      e = hipFuncSetAttribute((const void*)attn_bwd_dq_w64_kernel<D, RAGGED>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_dq_w64);
    return e;
  }();
  if (attr_status != hipSuccess) return KR_ELAUNCH;

  const int per = nq / nkv;
  const float scale_log2 = scale * kLog2e;
  const int dq_blocks = (sp / BQ) * nq * b;
  if (forms.shared_dq) {
    // 256-query tiles (see attn_forms): one wave per SIMD, 64 rows each.
    // It comes first: it also computes delta and the log2-domain copy of lse that the dK/dV kernel reads.
    hipLaunchKernelGGL((attn_bwd_dq_w64_kernel<D, RAGGED>), dim3(dq_blocks / 2), dim3(256), lds_dq_w64, st,
                       q, k, v, dout, o, lse,
                       neg_delta, neg_lse2, dq, s, nq, nkv, scale, scale_log2, ql, kl, vl, dol, ol, dql);
  } else {
    hipLaunchKernelGGL((attn_delta_kernel<D>), dim3((unsigned)((rows * (D / 8) + 255) / 256)), dim3(256), 0, st,
                       dout, o, lse, neg_delta, neg_lse2, s, sp, nq, per, rows, dol, ol);
  }
  if (hipGetLastError() != hipSuccess) return KR_ELAUNCH;
  const dim3 grid_kv((sp / 128) * (nq / hpw) * b * qsplit);
  hipLaunchKernelGGL(dkdv_kernel(partial), grid_kv, dim3(512), lds_dkdv, st, q, k, v, dout, neg_lse2,
                     neg_delta, dk, dv, part_k, part_v, s, nq, nkv, partial ? qsplit : 1, hpw, scale, scale_log2, ql, kl,
                     vl, dol, dkl, dvl);
  if (partial) {
    if (hipGetLastError() != hipSuccess) return KR_ELAUNCH;
    const int64_t total = (int64_t)b * nkv * s * (D / 8);
    hipLaunchKernelGGL((attn_group_reduce_kernel<D>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       st, part_k, part_v, dk, dv, s, sp,
                       nq / hpw, nkv, qsplit, total, dkl, dvl);
  }
  if (hipGetLastError() != hipSuccess) return KR_ELAUNCH;
  if (forms.shared_dq) return kr_launch_status();  // its dQ kernel ran in front of the dK/dV kernel
  if (dq_blocks <= 4 * 256) {  // few workgroups: the longest causal rows set the time
    hipLaunchKernelGGL((attn_bwd_dq_kernel<D, RAGGED, 2>), dim3(dq_blocks), dim3(512), 2 * lds_dq, st,
                       q, k, v, dout, lse,
                       neg_delta, dq, s, nq, nkv, scale, scale_log2, ql, kl, vl, dol,
                       dql);
  } else {
    hipLaunchKernelGGL((attn_bwd_dq_kernel<D, RAGGED, 1>), dim3(dq_blocks), dim3(256), lds_dq, st,
                       q, k, v, dout, lse,
                       neg_delta, dq, s, nq, nkv, scale, scale_log2, ql, kl, vl, dol,
                       dql);
  }
  return kr_launch_status();
}
}  // namespace

static int attn_bwd_impl(const void* dout, const void* q, const void* k, const void* v,
                           const void* o, const float* lse, void* dq, void* dk, void* dv,
                           void* workspace, int s, int b, int nq, int nkv, int hd, float scale,
                           int64_t q_ss, int64_t q_sb, int64_t q_sg, int64_t q_sh, int64_t k_ss,
                           int64_t k_sb, int64_t k_sh, int64_t v_ss, int64_t v_sb, int64_t v_sh,
                           int64_t o_ss, int64_t o_sb, int64_t o_sg, int64_t o_sh, int64_t do_ss,
                           int64_t do_sb, int64_t do_sg, int64_t do_sh, int64_t dq_ss, int64_t dq_sb,
                           int64_t dq_sg, int64_t dq_sh, int64_t dk_ss, int64_t dk_sb, int64_t dk_sh,
                           int64_t dv_ss, int64_t dv_sb, int64_t dv_sh, int flags, void* stream) {
  if (flags & ~(KR_ATTN_BESIDE_OTHER_STREAMS | KR_ATTN_GENERAL_KERNELS)) return KR_EINVAL;
  if (!dout || !q || !k || !v || !o || !lse || !dq || !dk || !dv || !workspace) return KR_EINVAL;
  const int rc = check_attn_common(s, b, nq, nkv, hd);
  if (rc != KR_OK) return rc;
  const void* ptrs[] = {dout, q, k, v, o, dq, dk, dv, workspace};
  for (const void* p : ptrs)
    if (!kr_aligned16(p)) return KR_EINVAL;
  if ((q_ss | q_sb | q_sg | q_sh | k_ss | k_sb | k_sh | v_ss | v_sb | v_sh | o_ss | o_sb | o_sg |
       o_sh | do_ss | do_sb | do_sg | do_sh | dq_ss | dq_sb | dq_sg | dq_sh | dk_ss | dk_sb |
       dk_sh | dv_ss | dv_sb | dv_sh) % 8)
    return KR_EINVAL;
  {
    const int64_t seq[] = {q_ss, k_ss, v_ss, o_ss, do_ss, dq_ss, dk_ss, dv_ss};
    if (!attn_strides_ok(seq, {q_sb, q_sg, q_sh, k_sb, k_sh, v_sb, v_sh, o_sb, o_sg, o_sh, do_sb, do_sg,
                               do_sh, dq_sb, dq_sg, dq_sh, dk_sb, dk_sh, dv_sb, dv_sh}))
      return KR_EUNSUPPORTED;
  }
  hipStream_t st = (hipStream_t)stream;
  const QLayout ql{q_ss, q_sb, q_sg, q_sh}, ol{o_ss, o_sb, o_sg, o_sh}, dol{do_ss, do_sb, do_sg, do_sh},
      dql{dq_ss, dq_sb, dq_sg, dq_sh};
  const KLayout kl{k_ss, k_sb, k_sh}, vl{v_ss, v_sb, v_sh}, dkl{dk_ss, dk_sb, dk_sh},
      dvl{dv_ss, dv_sb, dv_sh};
  float* delta = (float*)workspace;
  const bool in_place = attn_in_place(s, hd, {q_ss, k_ss, v_ss, o_ss, do_ss, dq_ss, dk_ss, dv_ss});
  if (!in_place && !(flags & KR_ATTN_GENERAL_KERNELS)) {
    // padded into the MFMA kernels: dO, q, o, k, v and the log-sum-exp go in, dq, dk, dv come back
    const int sp = attn_padded_len(s), per = nq / nkv;
    const size_t qb = attn_padded_bytes(s, b, nq), kb = attn_padded_bytes(s, b, nkv);
    char* w = (char*)workspace;
    void *do_p = w, *q_p = w + qb, *o_p = w + 2 * qb, *dq_p = w + 3 * qb;
    w += 4 * qb;
    void *k_p = w, *v_p = w + kb, *dk_p = w + 2 * kb, *dv_p = w + 3 * kb;
    w += 4 * kb;
    float* lse_p = (float*)w;
    w += attn_padded_stat_bytes(s, b, nq);
    int rc2 = launch_pad(dout, do_p, s, b, nq, per, hd, dol, st);
    if (rc2 == KR_OK) rc2 = launch_pad(q, q_p, s, b, nq, per, hd, ql, st);
    if (rc2 == KR_OK) rc2 = launch_pad(o, o_p, s, b, nq, per, hd, ol, st);
    if (rc2 == KR_OK) rc2 = launch_pad(k, k_p, s, b, nkv, 1, hd, as_qlayout(kl), st);
    if (rc2 == KR_OK) rc2 = launch_pad(v, v_p, s, b, nkv, 1, hd, as_qlayout(vl), st);
    // rows beyond s: exp2(x - 1.4e30) = 0 for every finite score, so they add nothing to dK and dV
    if (rc2 == KR_OK) rc2 = launch_resize_rows(lse, lse_p, (int64_t)b * nq, s, sp, 1e30f, st);
    if (rc2 != KR_OK) return rc2;
    const QLayout pq = padded_qlayout(b, nq, per);
    const KLayout pk = padded_klayout(b, nkv);
    rc2 = attn_bwd_impl(do_p, q_p, k_p, v_p, o_p, lse_p, dq_p, dk_p, dv_p, w, sp, b, nq, nkv, HD, scale, pq.s_, pq.b_,
                        pq.g_, pq.h_, pk.s_, pk.b_, pk.h_, pk.s_, pk.b_, pk.h_, pq.s_, pq.b_, pq.g_, pq.h_, pq.s_,
                        pq.b_, pq.g_, pq.h_, pq.s_, pq.b_, pq.g_, pq.h_, pk.s_, pk.b_, pk.h_, pk.s_, pk.b_, pk.h_,
                        flags, stream);
    if (rc2 != KR_OK) return rc2;
    rc2 = launch_unpad(dq_p, dq, s, b, nq, per, hd, dql, st);
    if (rc2 == KR_OK) rc2 = launch_unpad(dk_p, dk, s, b, nkv, 1, hd, as_qlayout(dkl), st);
    if (rc2 == KR_OK) rc2 = launch_unpad(dv_p, dv, s, b, nkv, 1, hd, as_qlayout(dvl), st);
    return rc2;
  }
  if (!attn_fast_path(s, hd) && (flags & KR_ATTN_GENERAL_KERNELS)) {
    using namespace general;
    const dim3 qgrid((s + GT - 1) / GT, nq, b), kgrid((s + GT - 1) / GT, nkv, b);
    hipLaunchKernelGGL(attn_general_delta_kernel, qgrid, dim3(GTHREADS), 0, st, (const bf16*)dout,
                       (const bf16*)o, delta, s, nq, nkv, hd, dol, ol);
    if (hipGetLastError() != hipSuccess) return KR_ELAUNCH;
    hipLaunchKernelGGL(attn_general_dkdv_kernel, kgrid, dim3(GTHREADS), 0, st, (const bf16*)q,
                       (const bf16*)k, (const bf16*)v, (const bf16*)dout, lse, (const float*)delta,
                       (bf16*)dk, (bf16*)dv, s, nq, nkv, hd, scale, ql, kl, vl, dol, dkl, dvl);
    if (hipGetLastError() != hipSuccess) return KR_ELAUNCH;
    hipLaunchKernelGGL(attn_general_dq_kernel, qgrid, dim3(GTHREADS), 0, st, (const bf16*)q,
                       (const bf16*)k, (const bf16*)v, (const bf16*)dout, lse, (const float*)delta,
                       (bf16*)dq, s, nq, nkv, hd, scale, ql, kl, vl, dol, dql);
    return kr_launch_status();
  }
  const BwdCall c{(const bf16*)dout, (const bf16*)q, (const bf16*)k, (const bf16*)v, (const bf16*)o, lse, (bf16*)dq,
                  (bf16*)dk, (bf16*)dv, delta, s, b, nq, nkv, scale, ql, ol, dol, dql, kl, vl, dkl, dvl, flags, st};
  if (hd == 64) return s % BQ ? attn_bwd_mfma<64, true>(c) : attn_bwd_mfma<64, false>(c);
  return s % BQ ? attn_bwd_mfma<128, true>(c) : attn_bwd_mfma<128, false>(c);
}

extern "C" int kr_attn_bwd(const void* dout, const void* q, const void* k, const void* v,
                           const void* o, const float* lse, void* dq, void* dk, void* dv,
                           void* workspace, int s, int b, int nq, int nkv, int hd, float scale,
                           int64_t q_ss, int64_t q_sb, int64_t q_sg, int64_t q_sh, int64_t k_ss,
                           int64_t k_sb, int64_t k_sh, int64_t v_ss, int64_t v_sb, int64_t v_sh,
                           int64_t o_ss, int64_t o_sb, int64_t o_sg, int64_t o_sh, int64_t do_ss,
                           int64_t do_sb, int64_t do_sg, int64_t do_sh, int64_t dq_ss, int64_t dq_sb,
                           int64_t dq_sg, int64_t dq_sh, int64_t dk_ss, int64_t dk_sb, int64_t dk_sh,
                           int64_t dv_ss, int64_t dv_sb, int64_t dv_sh, void* stream) {
  return attn_bwd_impl(dout, q, k, v, o, lse, dq, dk, dv, workspace, s, b, nq, nkv, hd, scale, q_ss, q_sb, q_sg,
                       q_sh, k_ss, k_sb, k_sh, v_ss, v_sb, v_sh, o_ss, o_sb, o_sg, o_sh, do_ss, do_sb, do_sg,
                       do_sh, dq_ss, dq_sb, dq_sg, dq_sh, dk_ss, dk_sb, dk_sh, dv_ss, dv_sb, dv_sh, 0, stream);
}

extern "C" int kr_attn_bwd_flags(const void* dout, const void* q, const void* k, const void* v,
                                 const void* o, const float* lse, void* dq, void* dk, void* dv,
                                 void* workspace, int s, int b, int nq, int nkv, int hd, float scale,
                                 int64_t q_ss, int64_t q_sb, int64_t q_sg, int64_t q_sh, int64_t k_ss,
                                 int64_t k_sb, int64_t k_sh, int64_t v_ss, int64_t v_sb, int64_t v_sh,
                                 int64_t o_ss, int64_t o_sb, int64_t o_sg, int64_t o_sh, int64_t do_ss,
                                 int64_t do_sb, int64_t do_sg, int64_t do_sh, int64_t dq_ss,
                                 int64_t dq_sb, int64_t dq_sg, int64_t dq_sh, int64_t dk_ss,
                                 int64_t dk_sb, int64_t dk_sh, int64_t dv_ss, int64_t dv_sb,
                                 int64_t dv_sh, int flags, void* stream) {
  return attn_bwd_impl(dout, q, k, v, o, lse, dq, dk, dv, workspace, s, b, nq, nkv, hd, scale, q_ss, q_sb, q_sg,
                       q_sh, k_ss, k_sb, k_sh, v_ss, v_sb, v_sh, o_ss, o_sb, o_sg, o_sh, do_ss, do_sb, do_sg,
                       do_sh, dq_ss, dq_sb, dq_sg, dq_sh, dk_ss, dk_sb, dk_sh, dv_ss, dv_sb, dv_sh, flags, stream);
}

namespace {
struct FwdCall {
  const bf16 *q, *k, *v;
  bf16* o;
  float* lse;
  int s, b, nq, nkv;
  float scale;
  QLayout ql, ol;
  KLayout kl, vl;
  int flags;
  hipStream_t st;
};

template <int D, bool RAGGED>
int attn_fwd_mfma(const FwdCall& c) {
  const int s = c.s, b = c.b, nq = c.nq, sp = attn_padded_len(s);
  if (attn_forms(sp, b, nq, c.nkv, D, c.flags).shared_fwd) {
    // 256-query tiles (see attn_forms): the halves share their K / V tiles
    constexpr size_t lds_sh = 3 * 16 * ((1024 + 16) + (1024 + 64));  // 100 KiB
    static const hipError_t attr_sh = hipFuncSetAttribute(
        (const void*)attn_fwd_sh_kernel<D, RAGGED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_sh);
    if (attr_sh != hipSuccess) return KR_ELAUNCH;
    hipLaunchKernelGGL((attn_fwd_sh_kernel<D, RAGGED>), dim3((sp / 256) * nq * b), dim3(512), lds_sh, c.st,
                       c.q, c.k, c.v, c.o, c.lse, s, c.nq, c.nkv, c.scale * kLog2e, c.ql.s_, c.ql.b_, c.ql.g_, c.ql.h_, c.kl.s_,
                       c.kl.b_, c.kl.h_, c.vl.s_, c.vl.b_, c.vl.h_, c.ol.s_, c.ol.b_, c.ol.g_, c.ol.h_);
    return kr_launch_status();
  }
  // two K and two V tiles of 17 KiB (padded blocks) per half; afterwards the same memory holds
  // the hand-over of half 1 (66 KiB) and, from 68 KiB on, 4 KiB of output staging per wave
  constexpr size_t lds_pp = 2 * 2 * 16 * ((1024 + 16) + (1024 + 64));  // 133 KiB
  static_assert(lds_pp >= 84 * 1024, "hand-over and output staging must fit");
  static const hipError_t attr_status = hipFuncSetAttribute(
      (const void*)attn_fwd_pp_kernel<D, RAGGED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_pp);
  if (attr_status != hipSuccess) return KR_ELAUNCH;
  hipLaunchKernelGGL((attn_fwd_pp_kernel<D, RAGGED>), dim3((sp / BQ) * nq * b), dim3(512), lds_pp, c.st,
                     c.q, c.k, c.v, c.o, c.lse, s, c.nq, c.nkv, c.scale * kLog2e, c.ql.s_, c.ql.b_, c.ql.g_, c.ql.h_, c.kl.s_,
                     c.kl.b_, c.kl.h_, c.vl.s_, c.vl.b_, c.vl.h_, c.ol.s_, c.ol.b_, c.ol.g_, c.ol.h_);
  return kr_launch_status();
}
}  // namespace

static int attn_fwd_impl(const void* q, const void* k, const void* v, void* o, float* lse, int s,
                           int b, int nq, int nkv, int hd, float scale, int64_t q_ss, int64_t q_sb,
                           int64_t q_sg, int64_t q_sh, int64_t k_ss, int64_t k_sb, int64_t k_sh,
                           int64_t v_ss, int64_t v_sb, int64_t v_sh, int64_t o_ss, int64_t o_sb,
                           int64_t o_sg, int64_t o_sh, int flags, void* stream, void* workspace = nullptr,
                           size_t workspace_bytes = 0) {
  if (flags & ~(KR_ATTN_BESIDE_OTHER_STREAMS | KR_ATTN_GENERAL_KERNELS | KR_ATTN_IN_PLACE)) return KR_EINVAL;
  if (!q || !k || !v || !o || !lse) return KR_EINVAL;
  if (workspace && !kr_aligned16(workspace)) return KR_EINVAL;
  const int rc = check_attn_common(s, b, nq, nkv, hd);
  if (rc != KR_OK) return rc;
  if (!kr_aligned16(q) || !kr_aligned16(k) || !kr_aligned16(v) || !kr_aligned16(o)) return KR_EINVAL;
  if ((q_ss | q_sb | q_sg | q_sh | k_ss | k_sb | k_sh | v_ss | v_sb | v_sh | o_ss | o_sb | o_sg |
       o_sh) % 8)
    return KR_EINVAL;
  {
    const int64_t seq[] = {q_ss, k_ss, v_ss, o_ss};
    if (!attn_strides_ok(seq, {q_sb, q_sg, q_sh, k_sb, k_sh, v_sb, v_sh, o_sb, o_sg, o_sh}))
      return KR_EUNSUPPORTED;
  }
  const bool in_place = attn_in_place(s, hd, {q_ss, k_ss, v_ss, o_ss});
  // Outside the training workloads' shapes a call without a workspace gets the general kernels, whose
  // probabilities stay fp32, also where the MFMA kernels (bf16 probabilities) would need no workspace.
  // (unless it asks for them: KR_ATTN_IN_PLACE)
  const bool asked_in_place = in_place && (flags & KR_ATTN_IN_PLACE) && !(flags & KR_ATTN_GENERAL_KERNELS);
  const bool general_kernels = !attn_fast_path(s, hd) && !asked_in_place &&
                               ((flags & KR_ATTN_GENERAL_KERNELS) || workspace == nullptr);
  // (a workspace that is there but too small is a caller's mistake, not a request for the general kernels)
  if (!attn_fast_path(s, hd) && !asked_in_place && !(flags & KR_ATTN_GENERAL_KERNELS) && workspace != nullptr &&
      workspace_bytes < kr_attn_fwd_workspace_bytes(s, b, nq, nkv, hd))
    return KR_EINVAL;
  if (!in_place && !general_kernels) {
    // padded into the MFMA kernels
    hipStream_t st = (hipStream_t)stream;
    const int sp = attn_padded_len(s), per = nq / nkv;
    const size_t qb = attn_padded_bytes(s, b, nq), kb = attn_padded_bytes(s, b, nkv);
    char* w = (char*)workspace;
    void *q_p = w, *o_p = w + qb, *k_p = w + 2 * qb, *v_p = w + 2 * qb + kb;
    float* lse_p = (float*)(w + 2 * qb + 2 * kb);
    const QLayout ql{q_ss, q_sb, q_sg, q_sh}, ol{o_ss, o_sb, o_sg, o_sh};
    const KLayout kl{k_ss, k_sb, k_sh}, vl{v_ss, v_sb, v_sh};
    int rc2 = launch_pad(q, q_p, s, b, nq, per, hd, ql, st);
    if (rc2 == KR_OK) rc2 = launch_pad(k, k_p, s, b, nkv, 1, hd, as_qlayout(kl), st);
    if (rc2 == KR_OK) rc2 = launch_pad(v, v_p, s, b, nkv, 1, hd, as_qlayout(vl), st);
    if (rc2 != KR_OK) return rc2;
    const QLayout pq = padded_qlayout(b, nq, per);
    const KLayout pk = padded_klayout(b, nkv);
    rc2 = attn_fwd_impl(q_p, k_p, v_p, o_p, lse_p, sp, b, nq, nkv, HD, scale, pq.s_, pq.b_, pq.g_, pq.h_, pk.s_, pk.b_,
                        pk.h_, pk.s_, pk.b_, pk.h_, pq.s_, pq.b_, pq.g_, pq.h_, flags, stream);
    if (rc2 != KR_OK) return rc2;
    rc2 = launch_unpad(o_p, o, s, b, nq, per, hd, ol, st);
    if (rc2 == KR_OK) rc2 = launch_resize_rows(lse_p, lse, (int64_t)b * nq, sp, s, 0.f, st);
    return rc2;
  }
  if (general_kernels) {
    using namespace general;
    const QLayout ql{q_ss, q_sb, q_sg, q_sh}, ol{o_ss, o_sb, o_sg, o_sh};
    const KLayout kl{k_ss, k_sb, k_sh}, vl{v_ss, v_sb, v_sh};
    hipLaunchKernelGGL(attn_general_fwd_kernel, dim3((s + GT - 1) / GT, nq, b), dim3(GTHREADS), 0,
                       (hipStream_t)stream, (const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)o,
                       lse, s, nq, nkv, hd, scale, ql, kl, vl, ol);
    return kr_launch_status();
  }
  const FwdCall c{(const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)o, lse, s, b, nq, nkv, scale,
                  QLayout{q_ss, q_sb, q_sg, q_sh}, QLayout{o_ss, o_sb, o_sg, o_sh}, KLayout{k_ss, k_sb, k_sh},
                  KLayout{v_ss, v_sb, v_sh}, flags, (hipStream_t)stream};
  if (hd == 64) return s % BQ ? attn_fwd_mfma<64, true>(c) : attn_fwd_mfma<64, false>(c);
  return s % BQ ? attn_fwd_mfma<128, true>(c) : attn_fwd_mfma<128, false>(c);
}

extern "C" int kr_attn_fwd(const void* q, const void* k, const void* v, void* o, float* lse, int s,
                           int b, int nq, int nkv, int hd, float scale, int64_t q_ss, int64_t q_sb,
                           int64_t q_sg, int64_t q_sh, int64_t k_ss, int64_t k_sb, int64_t k_sh,
                           int64_t v_ss, int64_t v_sb, int64_t v_sh, int64_t o_ss, int64_t o_sb,
                           int64_t o_sg, int64_t o_sh, void* stream) {
  return attn_fwd_impl(q, k, v, o, lse, s, b, nq, nkv, hd, scale, q_ss, q_sb, q_sg, q_sh, k_ss, k_sb, k_sh, v_ss,
                       v_sb, v_sh, o_ss, o_sb, o_sg, o_sh, 0, stream);
}

extern "C" int kr_attn_fwd_flags(const void* q, const void* k, const void* v, void* o, float* lse,
                                 int s, int b, int nq, int nkv, int hd, float scale, int64_t q_ss,
                                 int64_t q_sb, int64_t q_sg, int64_t q_sh, int64_t k_ss, int64_t k_sb,
                                 int64_t k_sh, int64_t v_ss, int64_t v_sb, int64_t v_sh, int64_t o_ss,
                                 int64_t o_sb, int64_t o_sg, int64_t o_sh, int flags, void* stream) {
  return attn_fwd_impl(q, k, v, o, lse, s, b, nq, nkv, hd, scale, q_ss, q_sb, q_sg, q_sh, k_ss, k_sb, k_sh, v_ss,
                       v_sb, v_sh, o_ss, o_sb, o_sg, o_sh, flags, stream);
}

// kr_attn_fwd_flags with a workspace of kr_attn_fwd_workspace_bytes(): a shape the MFMA kernels do not take as it
// lies (attn_in_place) is padded into them through the workspace; without one the general kernels take every shape but
// the training workloads', or, with KR_ATTN_IN_PLACE, every shape that would have to be padded.
extern "C" int kr_attn_fwd_ws(const void* q, const void* k, const void* v, void* o, float* lse, int s, int b,
                              int nq, int nkv, int hd, float scale, int64_t q_ss, int64_t q_sb, int64_t q_sg,
                              int64_t q_sh, int64_t k_ss, int64_t k_sb, int64_t k_sh, int64_t v_ss, int64_t v_sb,
                              int64_t v_sh, int64_t o_ss, int64_t o_sb, int64_t o_sg, int64_t o_sh, int flags,
                              void* workspace, size_t workspace_bytes, void* stream) {
  return attn_fwd_impl(q, k, v, o, lse, s, b, nq, nkv, hd, scale, q_ss, q_sb, q_sg, q_sh, k_ss, k_sb, k_sh, v_ss,
                       v_sb, v_sh, o_ss, o_sb, o_sg, o_sh, flags, stream, workspace, workspace_bytes);
}
