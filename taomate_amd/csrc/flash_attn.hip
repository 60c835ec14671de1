// Flash-style attention forward for gfx950 (CDNA4) over segmented keys.
//
// Replaces F.scaled_dot_product_attention as reached through
// standard_attention_forward (ltx_causal/attention/flex_attention_utils.py:225-276)
// from attention_with_cache (ltx_causal/transformer/kv_cache.py:1531), whose keys
// are torch.cat([cached_k, k], 1) (kv_cache.py:1487-1491).  Here the keys stay
// where they live (anchor | memory | window | current spans of a KV arena) and
// the kernel walks the spans in order.
//
// Work decomposition.  A workgroup of 4 wavefronts owns BM = 128 query rows of
// one (batch, head); each wavefront owns 32 rows.  Keys stream through LDS in
// tiles of BN = 64, double buffered: while the MFMAs consume tile j, the next
// tile is already in registers (global loads issued one tile ahead).
//
// Matrix-core mapping of the staged and fp8 kernels (v_mfma_f32_32x32x16_bf16,
// lane l, i = l % 32, g = l / 32; the bf16 pipelined kernel's 16x16x32 mapping
// stands at its body):
//   S^T = K Q^T: A = K rows (LDS), B = Q^T (registers, loaded once).  The
//   accumulator gives every lane ONE query (i) and 16 keys of each 32-key block,
//   so the softmax row statistics are per-lane scalars plus a single exchange
//   with lane l ^ 32, which holds the other 16 keys of the same query.
//   K rows are stored in LDS with row-index bits 2 and 3 swapped; with that
//   order accumulator register r of block kb holds key kb*32 + 16*(r/8) + 8g +
//   r%8, i.e. each lane's 8-register half is 8 consecutive keys.
//   O^T += V^T P^T: B = P straight from the softmax registers (8 consecutive
//   keys per lane, as above), A = V^T read from a transposed V tile in LDS.
//   The accumulator again gives each lane one query, so the online-softmax
//   rescale is one scalar per lane.
// Softmax: base-2 exponent with log2(e) folded into the logit scale
// (exp(x) = 2^(x*log2 e)), running max / running sum per query (the online
// normaliser of Milakov & Gimelshein 2018, as used by Dao et al. 2022).
// fp8 KV: tiles are decoded to bf16 on their way into LDS; the per-(head,
// frame) scales are folded into the logit scale (K) and into P (V).

#include <mutex>
#include <type_traits>

#include "ltx_common.h"

namespace ltx {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

struct FlashParams {
  const uint16_t* q;
  uint16_t* o;
  float* lse;
  const float* mask;
  int64_t q_bs, q_ls, q_hs;
  int64_t o_bs, o_ls, o_hs;
  int o_al16;                        // o and its strides are 16-byte aligned (staged output stores)
  int64_t kv_ls, kv_hs;              // K (and token-major V) token and head strides
  int64_t seg_bs[LTX_MAX_SEGMENTS];  // and each segment's batch stride, in bytes
  int64_t v_bs, v_hs, v_ds;          // key-major V: element (b, t, h, d) at b*v_bs + h*v_hs + d*v_ds + t
  int64_t sc_bs, sc_hs;
  int64_t mask_bs;
  int64_t Lk;
  // per-batch key counts (n_klen == B, or 0 for none): batch row b attends
  // keys [0, klen[b]) of the concatenated sequence (a key-padding mask that
  // keeps a prefix of each row)
  int n_klen;
  int klen[LTX_MAX_KEYLEN_BATCH];
  int64_t seg_start[LTX_MAX_SEGMENTS + 1];
  const void* k_ptr[LTX_MAX_SEGMENTS];
  const void* v_ptr[LTX_MAX_SEGMENTS];
  const float* k_sc[LTX_MAX_SEGMENTS];
  const float* v_sc[LTX_MAX_SEGMENTS];
  int tile_start[LTX_MAX_SEGMENTS + 1];  // first key tile of each segment (cumulative)
  int B, H, Lq, n_seg, n_qtiles, frame;
  // Balanced tail: the first n_full q-tiles run whole; each of the remaining
  // q-tiles is cut into `split` key ranges run by separate workgroups, whose
  // partial results meet in the workspace and are combined by a second kernel.
  int n_full, split;
  // pair kernel (bf16 key-major V, n_qtiles even): work unit u is q-tiles 2u
  // and 2u + 1, which lie in one (batch, head) and share every K/V tile;
  // n_full and split count units, and the tail q-tiles start at 2 n_full.
  int pair;
  void* part_o;    // [tail tiles * split][kBM][D] O / l of the key range (0 where l = 0), bf16 or
  int part_f32;    // float32 (see plan_split)
  float* part_ml;  // [tail tiles * split][kBM][2] running max (log2) and sum
  float scale;       // softmax scale applied to q.k
  float scale_log2;  // scale * log2(e)
};

// Max / sum of a lane's value with lane l ^ 32's (the lane holding the other
// 16 keys of the same query): one v_permlane32_swap, no LDS round trip.
__device__ __forceinline__ float pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The same over the four lanes l ^ 16, l ^ 32, l ^ 48 (the pipelined kernels'
// layout: a query's keys lie in four lanes).
__device__ __forceinline__ float quad_max(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return pair_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
__device__ __forceinline__ float quad_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return pair_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

// Which kernels can store float32 partials (FlashParams::part_f32): the launch
// plan asks no others for them.
constexpr bool stores_f32_partials(int D, bool pair, bool token) { return !pair || (token && D == 64); }

constexpr int kBM = 128;
constexpr int kBN = 64;
constexpr float kLog2e = 1.4426950408889634f;

// Row r of a K tile is stored at LDS row sig(r): bits 2 and 3 swapped.
__device__ __forceinline__ int sig(int r) { return (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1); }

// The pipelined kernels' tile layout in LDS: rows of NC 16-byte chunks without
// padding, chunk c of row r stored at c ^ row_swizzle(r), so that the 16 rows
// that a fragment read touches (one chunk index each) fall on 16 different
// 16-byte bank groups.  K rows hold keys in the order key_of_row: LDS row bits
// (half, kbit, g1 g0, r1 r0) hold key bits (half, g1 g0, kbit, r1 r0), so that
// a lane's scores of two adjacent 16-key blocks are 8 consecutive keys.
template <int NC>
__host__ __device__ constexpr int row_swizzle(int r) { return NC == 16 ? (r & 15) : ((r >> 1) & 7); }
// chunk pairs of a token-major V tile's key rows: the 8 keys that half a
// transposing fragment read touches (two blocks of 4, 8 keys apart, one 32-byte
// chunk pair each) fall on 8 different 32-byte bank groups
template <int NC>
__host__ __device__ constexpr int key_swizzle(int r) {
  return NC == 16 ? 2 * ((r & 3) | ((r >> 1) & 4)) : 2 * (((r >> 1) & 1) | ((r >> 2) & 2));
}
__host__ __device__ constexpr int key_of_row(int r) { return (r & 35) | ((r & 12) << 1) | ((r & 16) >> 2); }

// Blocks are dispatched round-robin over the 8 XCDs (block id % 8).  Give each
// XCD a contiguous range of the (batch*head, q-tile) space so the q-tiles that
// share one head's K/V run on the same XCD and hit the same L2.
__device__ __forceinline__ int xcd_remap(int bid, int nb) {
  const int xcd = bid & 7, slot = bid >> 3;
  const int per = nb >> 3, rem = nb & 7;
  return xcd * per + (xcd < rem ? xcd : rem) + slot;
}

template <bool FP8>
struct KVChunk;
template <>
struct KVChunk<false> {
  using raw_t = uint4;  // 8 bf16
  static __device__ __forceinline__ raw_t zero() { return make_uint4(0, 0, 0, 0); }
  static __device__ __forceinline__ raw_t load(const void* base, int64_t off) {
    return *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(base) + off);
  }
  static __device__ __forceinline__ raw_t bload(__amdgpu_buffer_rsrc_t r, int off) {
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    return make_uint4(v[0], v[1], v[2], v[3]);
  }
  static __device__ __forceinline__ uint4 to_bf16(raw_t r) { return r; }
};
template <>
struct KVChunk<true> {
  using raw_t = uint2;  // 8 fp8
  static __device__ __forceinline__ raw_t zero() { return make_uint2(0, 0); }
  static __device__ __forceinline__ raw_t load(const void* base, int64_t off) {
    return *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(base) + off);
  }
  static __device__ __forceinline__ raw_t bload(__amdgpu_buffer_rsrc_t r, int off) {
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
    return make_uint2(v[0], v[1]);
  }
  // Exact: every e4m3 value (subnormals included) is representable in bf16,
  // and v_cvt_scalef32_pk_bf16_fp8 with scale 1 decodes two codes (bytes 0-1
  // or 2-3 of the word) into a packed bf16 pair; its output was compared with
  // the e4m3 definition for every code pair on gfx950.
  static __device__ __forceinline__ uint32_t pair(uint32_t w, bool hi) {
    return __builtin_bit_cast(uint32_t, hi ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true)
                                           : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false));
  }
  static __device__ __forceinline__ uint4 to_bf16(raw_t r) {
    return make_uint4(pair(r.x, false), pair(r.x, true), pair(r.y, false), pair(r.y, true));
  }
};

// Key tiles never cross a segment: each segment is cut into ceil(len / kBN)
// tiles (the last one partial).  The iterator walks them in order with
// wave-uniform (scalar) state, touching the per-segment kernel arguments only
// when it enters a new segment.
struct TileIter {
  int s;
  int64_t row0;  // first token of the tile inside segment s
  int64_t len;   // tokens in segment s
  int64_t key0;  // first token of the tile in the concatenated key sequence
  const void* k;
  const void* v;

  __device__ __forceinline__ void enter(const FlashParams& p, int seg) {
    s = seg;
    row0 = 0;
    key0 = p.seg_start[seg];
    len = p.seg_start[seg + 1] - key0;
    k = p.k_ptr[seg];
    v = p.v_ptr[seg];
  }
  __device__ __forceinline__ void next(const FlashParams& p) {
    row0 += kBN;
    key0 += kBN;
    if (row0 >= len && s + 1 < p.n_seg) enter(p, s + 1);
  }
  __device__ __forceinline__ int nvalid() const {
    return (int)(len - row0 < kBN ? len - row0 : kBN);
  }
  // position on key tile j of the concatenated sequence
  __device__ __forceinline__ void seek(const FlashParams& p, int j) {
    int seg = 0;
    for (int i = 1; i < p.n_seg; ++i) seg = (j >= p.tile_start[i]) ? i : seg;
    enter(p, seg);
    row0 = (int64_t)(j - p.tile_start[seg]) * kBN;
    key0 += row0;
  }
};

// Key tiles of the concatenated sequence that hold keys below `lim` (the
// tiles a batch row with a per-batch key count attends; bf16 tiling).
__device__ __forceinline__ int tiles_below(const FlashParams& p, int lim) {
  int t = p.tile_start[p.n_seg];
  for (int i = p.n_seg - 1; i >= 0; --i)
    if (lim <= p.seg_start[i + 1]) {
      const int64_t in = lim - p.seg_start[i];
      t = p.tile_start[i] + (int)((in > 0 ? in : 0) + kBN - 1) / kBN;
    }
  return t;
}

// Which q-tile and key-tile range block `bid` owns.  Blocks below n_full take
// whole q-tiles; the rest take 1/split of a tail q-tile's key tiles.  Each
// group is spread over the 8 XCDs on its own (dispatch is round-robin by
// block id), and inside a group consecutive work shares an XCD's L2.
struct WorkItem {
  int qtile;   // linear (b*H + h) * n_qtiles + qt
  int j0, j1;  // key tiles [j0, j1)
  int piece;   // -1: whole q-tile; else index into the partial buffers
  int tail;    // tail q-tile index (piece >= 0)
};
__device__ __forceinline__ WorkItem work_item(const FlashParams& p, int bid, int ntiles) {
  WorkItem w;
  if (bid < p.n_full) {
    w.qtile = xcd_remap(bid, p.n_full);
    w.j0 = 0;
    w.j1 = ntiles;
    w.piece = -1;
    w.tail = -1;
  } else {
    const int ntail = gridDim.x - p.n_full;
    const int t = xcd_remap(bid - p.n_full, ntail);
    w.tail = t / p.split;
    const int part = t % p.split;
    w.qtile = p.n_full + w.tail;
    w.j0 = (int)((int64_t)ntiles * part / p.split);
    w.j1 = (int)((int64_t)ntiles * (part + 1) / p.split);
    w.piece = t;
  }
  return w;
}

// Work of group grp of pair workgroup `bid`: q-tile 2u + grp of unit u
// (units below n_full run whole, the rest 1/split of their key tiles; a
// split unit's two q-tiles are tail q-tiles 2 tu and 2 tu + 1).
__device__ __forceinline__ WorkItem pair_work(const FlashParams& p, int bid, int grp, int ntiles) {
  WorkItem w;
  int u;
  if (bid < p.n_full) {
    u = xcd_remap(bid, p.n_full);
    w.j0 = 0;
    w.j1 = ntiles;
    w.piece = -1;
    w.tail = -1;
  } else {
    const int ntail = gridDim.x - p.n_full;
    const int t = xcd_remap(bid - p.n_full, ntail);
    const int tu = t / p.split, part = t % p.split;
    u = p.n_full + tu;
    w.j0 = (int)((int64_t)ntiles * part / p.split);
    w.j1 = (int)((int64_t)ntiles * (part + 1) / p.split);
    w.tail = 2 * tu + grp;
    w.piece = w.tail * p.split + part;
  }
  w.qtile = 2 * u + grp;
  return w;
}

// Epilogue shared by the kernels: normalise and store a whole q-tile, or
// store a key range's partial result (O normalised by its own sum, in bf16 or, with
// MAYBE_F32 and where the launch plan says so, in float32; running max and
// sum).  oacc holds O^T fragments (lane: query li,
// d = db*32 + 8*(r/4) + 4*hg + r%4); m_run / l_tot are per query.
//
// stage (the pipelined kernels): this wave's 32 x (D + 8) bf16 region of LDS,
// free once every wave is past its last K/V tile.  The wave's 32 rows go
// through it so that each store writes 16 bytes per lane and a store
// instruction covers whole rows (four 256-byte rows at D = 128) instead of 16
// bytes of each of 32 rows 8 KB apart: an eighth of the memory requests.
// The stores are streaming ones (whole rows now, so they leave the L2 as
// full lines while the kernel runs): 156.3 -> 154.0 us for the staging and
// 152.6 us with streaming stores at the 1152 x 4608 chunk, and the launch
// after it 1.5 us faster.  Every wave of the workgroup calls it (two
// barriers inside), with one path for the whole workgroup (a whole q-tile or
// a key range, and o_al16).
template <int D, bool MAYBE_F32>
__device__ __forceinline__ void finish_tile(const FlashParams& p, const WorkItem& w, int b, int h,
                                            int qt, int row, const f32x16_t (&oacc)[D / 32], float m_run,
                                            float l_tot, uint16_t* stage = nullptr) {
  constexpr int DB = D / 32;
  const int hg = (threadIdx.x & 63) >> 5;  // row: this lane's query inside the q-tile
  const int qi = qt * kBM + row;
  if (MAYBE_F32 && w.piece >= 0 && p.part_f32) {
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    float* po = static_cast<float*>(p.part_o) + ((int64_t)w.piece * kBM + row) * D + 4 * hg;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4)
        *reinterpret_cast<float4*>(po + d * 32 + 8 * g4) =
            make_float4(oacc[d][4 * g4] * inv, oacc[d][4 * g4 + 1] * inv, oacc[d][4 * g4 + 2] * inv,
                        oacc[d][4 * g4 + 3] * inv);
    if (hg == 0) *reinterpret_cast<float2*>(p.part_ml + ((int64_t)w.piece * kBM + row) * 2) = make_float2(m_run, l_tot);
    return;
  }
  if (stage != nullptr && (w.piece >= 0 || p.o_al16)) {
    constexpr int RS = D + 8;   // staging row stride (elements)
    constexpr int CPR = D / 8;  // 16-byte chunks per row
    const int li = threadIdx.x & 31, lane = threadIdx.x & 63;
    const int row0 = row - li;  // the wave's first row in the q-tile
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    __syncthreads();  // every wave is done reading the K/V tiles
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        uint2 v;
        v.x = pack_bf16x2(oacc[d][4 * g4] * inv, oacc[d][4 * g4 + 1] * inv);
        v.y = pack_bf16x2(oacc[d][4 * g4 + 2] * inv, oacc[d][4 * g4 + 3] * inv);
        *reinterpret_cast<uint2*>(stage + li * RS + d * 32 + 8 * g4 + 4 * hg) = v;
      }
    __syncthreads();
    if (w.piece < 0) {
      const int64_t obase = b * p.o_bs + h * p.o_hs;
#pragma unroll
      for (int i = 0; i < D / 16; ++i) {
        const int c = i * 64 + lane, r = c / CPR, cc = c % CPR;
        const int q = qt * kBM + row0 + r;
        const uint4 v = *reinterpret_cast<const uint4*>(stage + r * RS + cc * 8);
        if (q < p.Lq) store_stream(p.o + obase + (int64_t)q * p.o_ls + cc * 8, v);
      }
      if (p.lse != nullptr && hg == 0 && qi < p.Lq)
        p.lse[((int64_t)b * p.H + h) * p.Lq + qi] = (m_run + __log2f(l_tot)) / kLog2e;
    } else {
      uint16_t* po = static_cast<uint16_t*>(p.part_o) + ((int64_t)w.piece * kBM + row0) * D;
#pragma unroll
      for (int i = 0; i < D / 16; ++i) {
        const int c = i * 64 + lane, r = c / CPR, cc = c % CPR;
        store_stream(po + r * D + cc * 8, *reinterpret_cast<const uint4*>(stage + r * RS + cc * 8));
      }
      if (hg == 0) *reinterpret_cast<float2*>(p.part_ml + ((int64_t)w.piece * kBM + row) * 2) = make_float2(m_run, l_tot);
    }
    return;
  }
  if (w.piece < 0) {
    if (qi < p.Lq) {
      const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
      uint16_t* op = p.o + b * p.o_bs + (int64_t)qi * p.o_ls + h * p.o_hs;
#pragma unroll
      for (int d = 0; d < DB; ++d) {
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          uint2 v;
          v.x = pack_bf16x2(oacc[d][4 * g4] * inv, oacc[d][4 * g4 + 1] * inv);
          v.y = pack_bf16x2(oacc[d][4 * g4 + 2] * inv, oacc[d][4 * g4 + 3] * inv);
          *reinterpret_cast<uint2*>(op + d * 32 + 8 * g4 + 4 * hg) = v;
        }
      }
      if (p.lse != nullptr && hg == 0) p.lse[((int64_t)b * p.H + h) * p.Lq + qi] = (m_run + __log2f(l_tot)) / kLog2e;
    }
    return;
  }
  // ---- partial result of one key range: combined by flash_combine_kernel.
  // O is stored normalised by the range's own sum and rounded to bf16 (the
  // output's precision), half the bytes of float32; the combine weighs each
  // range by its sum and maximum. ----
  uint16_t* po = static_cast<uint16_t*>(p.part_o) + ((int64_t)w.piece * kBM + row) * D;
  const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      uint2 v;
      v.x = pack_bf16x2(oacc[d][4 * g4] * inv, oacc[d][4 * g4 + 1] * inv);
      v.y = pack_bf16x2(oacc[d][4 * g4 + 2] * inv, oacc[d][4 * g4 + 3] * inv);
      *reinterpret_cast<uint2*>(po + d * 32 + 8 * g4 + 4 * hg) = v;
    }
  if (hg == 0) *reinterpret_cast<float2*>(p.part_ml + ((int64_t)w.piece * kBM + row) * 2) = make_float2(m_run, l_tot);
}

// Epilogue of the pipelined kernels: normalise and store a wave's 32 rows of
// a whole q-tile, or store a key range's partial result (as finish_tile).  oacc[d][n] holds O^T fragments (lane: query
// row0 + 16 n + li, channels 16 d + 4 lg + r); m_run / l_tot are per query.
//
// stage: this wave's 32 x D bf16 region of LDS, free once every wave is past
// its last K/V tile.  The wave's rows go through it (16-byte chunks xor-swizzled
// by row, as the tiles) so that each store writes 16 bytes per lane and a
// store instruction covers whole rows (four 256-byte rows at D = 128) instead
// of 8 bytes of each of 16 rows 8 KB apart: an eighth of the memory requests.
// The stores are streaming ones (whole rows, so they leave the L2 as full
// lines while the kernel runs): 156.3 -> 154.0 us for the staging and
// 152.6 us with streaming stores at the 1152 x 4608 chunk, and the launch
// after it 1.5 us faster.  Every wave of the workgroup calls it (two
// barriers inside), with one path for the whole workgroup (a whole q-tile or
// a key range, part_f32 and o_al16).  Float32 partials go straight from the
// accumulators, 16 bytes per lane.
template <int D, bool MAYBE_F32>
__device__ __forceinline__ void finish_rows(const FlashParams& p, const WorkItem& w, int b, int h, int qt, int row0,
                                            const f32x4_t (&oacc)[D / 16][2], const float (&m_run)[2],
                                            const float (&l_tot)[2], uint16_t* stage) {
  constexpr int CPR = D / 8;  // 16-byte chunks per row
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const float inv[2] = {l_tot[0] > 0.0f ? 1.0f / l_tot[0] : 0.0f, l_tot[1] > 0.0f ? 1.0f / l_tot[1] : 0.0f};
  auto packed = [&](int d, int n) {
    return make_uint2(pack_bf16x2(oacc[d][n][0] * inv[n], oacc[d][n][1] * inv[n]),
                      pack_bf16x2(oacc[d][n][2] * inv[n], oacc[d][n][3] * inv[n]));
  };
  if (MAYBE_F32 && w.piece >= 0 && p.part_f32) {
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      float* po = static_cast<float*>(p.part_o) + ((int64_t)w.piece * kBM + row0 + 16 * n + li) * D + 4 * lg;
#pragma unroll
      for (int d = 0; d < D / 16; ++d) *reinterpret_cast<f32x4_t*>(po + d * 16) = oacc[d][n] * inv[n];
    }
  } else if (w.piece < 0 && !p.o_al16) {  // output rows that are only 8-byte aligned
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int qi = qt * kBM + row0 + 16 * n + li;
      if (qi >= p.Lq) continue;
      uint16_t* op = p.o + b * p.o_bs + (int64_t)qi * p.o_ls + h * p.o_hs + 4 * lg;
#pragma unroll
      for (int d = 0; d < D / 16; ++d) *reinterpret_cast<uint2*>(op + d * 16) = packed(d, n);
    }
  } else {
    __syncthreads();  // every wave is done reading the K/V tiles
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int d = 0; d < D / 16; ++d)
        *reinterpret_cast<uint2*>(stage + (16 * n + li) * D + ((2 * d + (lg >> 1)) ^ row_swizzle<CPR>(li)) * 8 +
                                  (lg & 1) * 4) = packed(d, n);
    __syncthreads();
    const int64_t obase = b * p.o_bs + h * p.o_hs;
    uint16_t* po = w.piece < 0 ? nullptr : static_cast<uint16_t*>(p.part_o) + ((int64_t)w.piece * kBM + row0) * D;
#pragma unroll
    for (int i = 0; i < D / 16; ++i) {
      const int c = i * 64 + lane, r = c / CPR, cc = c % CPR;
      const uint4 v = *reinterpret_cast<const uint4*>(stage + r * D + (cc ^ row_swizzle<CPR>(r & 15)) * 8);
      const int q = qt * kBM + row0 + r;
      if (po != nullptr)
        store_stream(po + r * D + cc * 8, v);
      else if (q < p.Lq)
        store_stream(p.o + obase + (int64_t)q * p.o_ls + cc * 8, v);
    }
  }
  if (lg != 0) return;
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int row = row0 + 16 * n + li, qi = qt * kBM + row;
    if (w.piece >= 0)
      *reinterpret_cast<float2*>(p.part_ml + ((int64_t)w.piece * kBM + row) * 2) = make_float2(m_run[n], l_tot[n]);
    else if (p.lse != nullptr && qi < p.Lq)
      p.lse[((int64_t)b * p.H + h) * p.Lq + qi] = (m_run[n] + __log2f(l_tot[n])) / kLog2e;
  }
}

constexpr int kMaxSplit = 8;  // key ranges a tail q-tile may be cut into

// Combines the `split` partial results of every tail q-tile, launched after the
// attention kernel on the same stream: out = sum_i w_i o_i / sum_i w_i with
// w_i = l_i 2^(m_i - max m) and o_i the range's normalised output (F32: in
// float32).  One thread per (query row, 8 output columns): every piece's (max,
// sum) and 16- or 32-byte O chunk are loaded up front, so each thread waits for one round of loads.
// The output is written as two 8-byte halves (the entry point guarantees
// 8-byte aligned output rows); the workspace partials are 16-byte aligned.
constexpr int kCombineCols = 8;
template <int D>
constexpr int combine_wg_per_tile() { return kBM / (256 / (D / kCombineCols)); }

template <int D, bool F32>
__global__ void __launch_bounds__(256) flash_combine_kernel(const FlashParams p) {
  constexpr int CG = D / kCombineCols;  // 8-column groups per row
  constexpr int ROWS = 256 / CG;        // rows per workgroup
  constexpr int WG_PER_TILE = kBM / ROWS;
  static_assert(WG_PER_TILE == combine_wg_per_tile<D>() && ROWS * WG_PER_TILE == kBM, "combine grid");
  const int tail = blockIdx.x / WG_PER_TILE;
  const int r = (blockIdx.x % WG_PER_TILE) * ROWS + threadIdx.x / CG;
  const int cg = threadIdx.x % CG;
  const int qtile = (p.pair ? 2 * p.n_full : p.n_full) + tail;
  const int qt = qtile % p.n_qtiles;
  const int bh = qtile / p.n_qtiles;
  const int b = bh / p.H, h = bh % p.H;
  const int q = qt * kBM + r;
  if (q >= p.Lq) return;
  const int64_t first = (int64_t)tail * p.split;
  f32x2_t ml[kMaxSplit];
  typedef std::conditional_t<F32, float, uint16_t> part_t;
  constexpr int CW = kCombineCols * sizeof(part_t) / 16;  // 16-byte words of a chunk
  uint4 o[kMaxSplit][CW];
#pragma unroll
  for (int i = 0; i < kMaxSplit; ++i) {
    if (i < p.split) {
      ml[i] = *reinterpret_cast<const f32x2_t*>(p.part_ml + ((first + i) * kBM + r) * 2);
      const part_t* po = static_cast<const part_t*>(p.part_o) + ((first + i) * kBM + r) * D + cg * kCombineCols;
#pragma unroll
      for (int c = 0; c < CW; ++c) o[i][c] = reinterpret_cast<const uint4*>(po)[c];
    }
  }
  float mmax = -INFINITY;
#pragma unroll
  for (int i = 0; i < kMaxSplit; ++i)
    if (i < p.split) mmax = fmaxf(mmax, ml[i][0]);
  float lsum = 0.0f;
  float acc[kCombineCols] = {};
#pragma unroll
  for (int i = 0; i < kMaxSplit; ++i) {
    if (i < p.split) {
      const float wgt = ml[i][0] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml[i][0] - mmax) * ml[i][1];
      lsum += wgt;
#pragma unroll
      for (int c = 0; c < CW; ++c) {
        const uint32_t w[4] = {o[i][c].x, o[i][c].y, o[i][c].z, o[i][c].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (F32) {
            acc[4 * c + e] += wgt * __uint_as_float(w[e]);
          } else {
            acc[2 * e] += wgt * bf16_bits_to_f32(w[e] & 0xFFFFu);
            acc[2 * e + 1] += wgt * bf16_bits_to_f32(w[e] >> 16);
          }
        }
      }
    }
  }
  const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;
  uint16_t* dst = p.o + b * p.o_bs + (int64_t)q * p.o_ls + h * p.o_hs + cg * kCombineCols;
  *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(acc[0] * inv, acc[1] * inv),
                                              pack_bf16x2(acc[2] * inv, acc[3] * inv));
  *reinterpret_cast<uint2*>(dst + 4) = make_uint2(pack_bf16x2(acc[4] * inv, acc[5] * inv),
                                                  pack_bf16x2(acc[6] * inv, acc[7] * inv));
  if (p.lse != nullptr && cg == 0) p.lse[((int64_t)b * p.H + h) * p.Lq + q] = (mmax + __log2f(lsum)) / kLog2e;
}

// Register-staged kernel for calls with an additive key mask (bf16, token-major
// V): the mask joins the logits, so the softmax takes every tile's maximum.
template <int D>
__global__ void __launch_bounds__(256, 2) flash_fwd_masked_kernel(const FlashParams p) {
  constexpr int BM = kBM, BN = kBN;
  constexpr int KS = D + 8;                // K tile LDS row stride (elements)
  constexpr int VS = BN + 8;               // V^T tile LDS row stride
  constexpr int KBUF = BN * KS;
  constexpr int VBUF = D * VS;
  constexpr int NKC = D / 8;               // 8-element chunks per K row
  constexpr int KROWS_PER_PASS = 256 / NKC;
  constexpr int K_LOADS = BN / KROWS_PER_PASS;
  constexpr int NVP = (BN / 4) * (D / 8);  // (4-key group, 8-d chunk) pairs
  constexpr int DB = D / 32;
  constexpr int QS = D / 16;
  using Chunk = KVChunk<false>;
  using raw_t = typename Chunk::raw_t;

  __shared__ __attribute__((aligned(16))) uint16_t smem[2 * (KBUF + VBUF)];
  __shared__ float mask_s[2][BN];

  const WorkItem wi = work_item(p, blockIdx.x, p.tile_start[p.n_seg]);
  const int qt = wi.qtile % p.n_qtiles;
  const int bh = wi.qtile / p.n_qtiles;
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int li = lane & 31, hg = lane >> 5;
  const int qi = qt * BM + wave * 32 + li;
  const int ntiles = wi.j1 - wi.j0;

  // ---- Q^T fragments, resident for the whole key loop ----
  bf16x8_t qf[QS];
  {
    const bool ok = qi < p.Lq;
    const uint16_t* qp = p.q + b * p.q_bs + (int64_t)(ok ? qi : 0) * p.q_ls + h * p.q_hs + hg * 8;
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      uint4 v = ok ? *reinterpret_cast<const uint4*>(qp + s * 16) : make_uint4(0, 0, 0, 0);
      qf[s] = __builtin_bit_cast(bf16x8_t, v);
    }
  }

  const int64_t kv_off = h * p.kv_hs;
  // rows this thread moves in every tile, as loop-invariant byte offsets from
  // the tile's first row (buffer loads return 0 past the tile's valid rows)
  const int kc = tid % NKC;
  const int kr0 = tid / NKC;
  const int vkg = tid % 16, vdc = tid / 16;
  const bool vthread = tid < NVP;
  constexpr int ESZ = 2;
  const int row_bytes = (int)(p.kv_ls * ESZ);
  int koff[K_LOADS], voff[4];
#pragma unroll
  for (int i = 0; i < K_LOADS; ++i) koff[i] = (kr0 + i * KROWS_PER_PASS) * row_bytes + kc * 8 * ESZ;
#pragma unroll
  for (int e = 0; e < 4; ++e) voff[e] = (vkg * 4 + e) * row_bytes + vdc * 8 * ESZ;

  // ---- global -> register prefetch of one K/V tile ----
  raw_t kreg[K_LOADS];
  raw_t vreg[4];
  float mreg = 0.0f;
  TileIter ld;
  ld.seek(p, wi.j0);
  auto load_tile = [&]() {
    const int64_t base = b * p.seg_bs[ld.s] + (kv_off + ld.row0 * p.kv_ls) * ESZ;
    const int nbytes = ld.nvalid() * row_bytes;
    const auto kr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(reinterpret_cast<const char*>(ld.k) + base), (short)0, nbytes, 0x00020000);
    const auto vr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(reinterpret_cast<const char*>(ld.v) + base), (short)0, nbytes, 0x00020000);
#pragma unroll
    for (int i = 0; i < K_LOADS; ++i) kreg[i] = Chunk::bload(kr, koff[i]);
    if (vthread) {
#pragma unroll
      for (int e = 0; e < 4; ++e) vreg[e] = Chunk::bload(vr, voff[e]);
    }
    if (tid < BN) mreg = tid < ld.nvalid() ? p.mask[b * p.mask_bs + ld.key0 + tid] : 0.0f;
    ld.next(p);
  };

  // ---- register -> LDS store (K rows permuted, V transposed) ----
  auto store_tile = [&](int buf) {
    uint16_t* ks = smem + buf * (KBUF + VBUF);
    uint16_t* vs = ks + KBUF;
#pragma unroll
    for (int i = 0; i < K_LOADS; ++i) {
      const int r = kr0 + i * KROWS_PER_PASS;
      *reinterpret_cast<uint4*>(ks + sig(r) * KS + kc * 8) = Chunk::to_bf16(kreg[i]);
    }
    if (vthread) {
      uint4 v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = Chunk::to_bf16(vreg[e]);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint32_t a0 = (&v[0].x)[w], a1 = (&v[1].x)[w], a2 = (&v[2].x)[w], a3 = (&v[3].x)[w];
        // d = vdc*8 + 2w (low halves) and 2w+1 (high halves); keys vkg*4 .. +3
        uint2 lo, hi;
        lo.x = __builtin_amdgcn_perm(a1, a0, 0x05040100u);
        lo.y = __builtin_amdgcn_perm(a3, a2, 0x05040100u);
        hi.x = __builtin_amdgcn_perm(a1, a0, 0x07060302u);
        hi.y = __builtin_amdgcn_perm(a3, a2, 0x07060302u);
        *reinterpret_cast<uint2*>(vs + (vdc * 8 + 2 * w) * VS + vkg * 4) = lo;
        *reinterpret_cast<uint2*>(vs + (vdc * 8 + 2 * w + 1) * VS + vkg * 4) = hi;
      }
    }
    if (tid < BN) mask_s[buf][tid] = mreg;
  };

  f32x16_t oacc[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d) oacc[d] = f32x16_t{};
  // Running max in the base-2 logit domain.  It is only raised when a new
  // maximum exceeds it by more than kLazy (then O and l are rescaled); in
  // between, P = 2^(x - m) may reach 2^kLazy, which float32 sums and bf16 P
  // represent exactly enough.  Exact: O and l always share the same m.
  constexpr float kLazy = 8.0f;
  float m_run = -INFINITY;
  float l_run = 0.0f;  // sum over this lane's 16-key halves

  if (ntiles > 0) {
    load_tile();
    store_tile(0);
    if (ntiles > 1) load_tile();
    __syncthreads();
  }
  TileIter cp;
  cp.seek(p, wi.j0);

  for (int j = 0; j < ntiles; ++j) {
    const int buf = j & 1;
    if (j + 1 < ntiles) {
      store_tile(buf ^ 1);
      if (j + 2 < ntiles) load_tile();
    }
    const uint16_t* ks = smem + buf * (KBUF + VBUF);
    const uint16_t* vs = ks + KBUF;
    const int nvalid = cp.nvalid();

    // ---- S^T = K Q^T, fragments read one k-step ahead ----
    f32x16_t sacc[2] = {f32x16_t{}, f32x16_t{}};
    const uint16_t* kfrag = ks + li * KS + hg * 8;
    bf16x8_t a0 = *reinterpret_cast<const bf16x8_t*>(kfrag);
    bf16x8_t a1 = *reinterpret_cast<const bf16x8_t*>(kfrag + 32 * KS);
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      bf16x8_t n0 = a0, n1 = a1;
      if (s + 1 < QS) {
        n0 = *reinterpret_cast<const bf16x8_t*>(kfrag + (s + 1) * 16);
        n1 = *reinterpret_cast<const bf16x8_t*>(kfrag + 32 * KS + (s + 1) * 16);
      }
      sacc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, qf[s], sacc[0], 0, 0, 0);
      sacc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, qf[s], sacc[1], 0, 0, 0);
      a0 = n0;
      a1 = n1;
    }
    // first V^T fragments, in flight during the softmax
    const uint16_t* vfrag = vs + li * VS + hg * 8;
    bf16x8_t va = *reinterpret_cast<const bf16x8_t*>(vfrag);
    bf16x8_t vb = *reinterpret_cast<const bf16x8_t*>(vfrag + 16);

    // ---- online softmax on the accumulators (base-2 domain) ----
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = kb * 32 + 16 * (r >> 3) + 8 * hg + (r & 7);
        sacc[kb][r] = fmaxf((sacc[kb][r] * p.scale + mask_s[buf][key]) * kLog2e, -3.0e38f);
      }
    if (nvalid < BN) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kb * 32 + 16 * (r >> 3) + 8 * hg + (r & 7);
          if (key >= nvalid) sacc[kb][r] = -INFINITY;
        }
    }
    float mt = sacc[0][0];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, sacc[kb][r]);
    mt = pair_max(mt);
    const float m_tile = mt;
    const bool raise = m_tile > m_run + kLazy;
    if (__builtin_amdgcn_ballot_w64(raise)) {
      const float m_new = fmaxf(m_run, m_tile);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);  // 0 on the first tile
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < DB; ++d) oacc[d] *= alpha;
    }
    // all keys masked so far: keep the exponent finite
    const float neg_m = (m_run == -INFINITY) ? 0.0f : -m_run;

    float psum = 0.0f;
    bf16x8_t pf[4];
#pragma unroll
    for (int ks4 = 0; ks4 < 4; ++ks4) {
      const int kb = ks4 >> 1, t = ks4 & 1;
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float p0 = __builtin_amdgcn_exp2f(sacc[kb][8 * t + e] + neg_m);
        const float p1 = __builtin_amdgcn_exp2f(sacc[kb][8 * t + e + 1] + neg_m);
        psum += p0 + p1;
        w[e >> 1] = pack_bf16x2(p0, p1);
      }
      pf[ks4] = __builtin_bit_cast(bf16x8_t, make_uint4(w[0], w[1], w[2], w[3]));
    }
    l_run += psum;

    // ---- O^T += V^T P^T, fragments read one step ahead ----
#pragma unroll
    for (int d = 0; d < DB; ++d) {
#pragma unroll
      for (int ks4 = 0; ks4 < 4; ks4 += 2) {
        bf16x8_t na = va, nb = vb;
        const int nd = (ks4 + 2 < 4) ? d : d + 1;
        const int nk = (ks4 + 2 < 4) ? ks4 + 2 : 0;
        if (nd < DB) {
          na = *reinterpret_cast<const bf16x8_t*>(vfrag + nd * 32 * VS + nk * 16);
          nb = *reinterpret_cast<const bf16x8_t*>(vfrag + nd * 32 * VS + (nk + 1) * 16);
        }
        oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pf[ks4], oacc[d], 0, 0, 0);
        oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vb, pf[ks4 + 1], oacc[d], 0, 0, 0);
        va = na;
        vb = nb;
      }
    }
    cp.next(p);
    __syncthreads();
  }

  // ---- epilogue: combine the two lane halves' sums, then store or publish ----
  finish_tile<D, false>(p, wi, b, h, qt, (int)(threadIdx.x >> 6) * 32 + (int)(threadIdx.x & 31), oacc, m_run,
                 pair_sum(l_run));
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// ---------------------------------------------------------------------------
// Software-pipelined direct kernel (bf16; K token-major, V key- or token-major).
//
// What bounds it: power.  Under this kernel's random data the part clocks
// down to 1.6-1.8 GHz: the 32x32x16 form of the kernel took 157 us (151-164 by box) at
// 1152 x 4608 (B = 2, 32 heads x 128) and 106 us, the same instructions, on
// all-zero q, K and V.  So the matrix work runs on
// v_mfma_f32_16x16x32_bf16, which does the same FLOPs for less energy: a
// register-and-LDS loop with one 1 KB fragment read per 32 MFMA cycles
// sustains 1820 TFLOP/s on random data with it against 1593 with
// v_mfma_f32_32x32x16_bf16 (2364 and 2387 on zeros).  The kernel then takes
// 116 us on zeros (twice the MFMA issues and operand reads) but less on
// random data: 151.5 -> 144.3 us at 1152 queries and 211 -> 201.5 us at 1536
// on one box, back to back; with the norm + RoPE + append launch before it and
// K/V out of cache 184.8 -> 181.2 us.
//
// Matrix-core mapping (lane l, i = l % 16, g = l / 16): a wave owns 32
// queries as two blocks of 16, so every fragment read from LDS feeds two
// MFMAs.  S^T = K Q^T gives each lane one query per block and 4 keys of each
// 16-key block; with the K rows in key_of_row order two adjacent blocks'
// scores are 8 consecutive keys, the B operand of O^T += V^T P^T, so P goes
// from the exp registers into the product without a shuffle.  A query's
// keys lie in four lanes: statistics meet by quad_max / quad_sum.
//
// K and V^T tiles go HBM -> LDS with buffer_load ... lds (gfx950 writes 16
// bytes per lane straight into LDS: lane L of an instruction lands at base +
// 16*L), so no VGPRs and no VALU work go into staging.  Tile rows are not
// padded; the chunks of a row are xor-swizzled (row_swizzle) and the K-row
// order, the swizzle and the V transpose all happen in the address each lane
// reads from.  V stored key-major (the KV arena's layout): a segment's last
// 8-token chunk is read whole and its keys past the segment end are masked
// out of the softmax.  V stored token-major (VTOK: plain cache tensors): its
// tiles keep keys in rows and ds_read_b64_tr_b16 transposes the fragments, at
// about 158 against 147 us at 1152 x 4608, where concatenating K and copying
// V into a key-major store first took 105 us.
//
// The per-tile vector work is cut down and moved under the matrix cores:
//
// * P = 2^(S*c - m) (c = scale*log2 e) is one v_fma and one v_exp per score:
//   no tile maximum is taken on the common path.
// * The row sum (fp32 adds of the P values) doubles as the overflow check:
//   m is not raised every tile.  While the per-lane sum of a tile stays at or below 2^16, every P
//   of that tile is at most 2^16, which fp32 sums and bf16 P carry as exactly
//   as P <= 1.  When a lane's sum goes above it, the tile maximum is taken
//   and m, O and l are rescaled before P is redone (the online normaliser of
//   Milakov & Gimelshein 2018).  The first tile sets m from its own maximum,
//   so the sums never underflow.  Logits stay fp32-exact (Q is not rescaled).
// * Pipeline: iteration j computes O += V(j-1)^T P(j-1) on the matrix cores
//   while the vector unit turns S(j) into P(j), then S(j+1) = K(j+1) Q^T.
//   K is loaded two tiles ahead and V one tile ahead of their use; one
//   barrier per tile frees the buffers read in the previous iteration.
//
// fp8 K/V (token-major e4m3 codes with per-(batch, head, frame) scales) use
// the same slot program (tiles cut at frame boundaries, see KeyStreamT) on
// v_mfma_f32_32x32x16_bf16 and padded tile rows.  Decoded codes carry three
// mantissa bits, so their products cost less power (243 us at 1152 x 6912
// against 200 us on zeros) and the staging's issue cycles count instead: the
// 16x16x32 form measured 244 against 240 us.  The tiles are staged through
// registers:
// each thread loads 8-byte chunks of the next tiles from HBM one iteration
// ahead, and decodes them (exactly) to bf16 into the LDS buffers the barrier
// freed, K rows in the swapped order and V transposed with v_perm, so every
// code is decoded once per workgroup.  The decode and the next loads are
// spread over the slot program of the tile, under its matrix work.  A tile never crosses a frame
// (KeyStreamT<true>), so its scales are two scalars: the K scale joins
// the logit scale, c_j = c * sk_j, and the V scale joins the exponent,
// P' = 2^(S c_j - m + log2 sv_j) = sv_j P, so the PV MFMAs read plain codes;
// the row sum and the overflow check use sum(P') / sv_j.
// ---------------------------------------------------------------------------

// One operand (K or V) of the concatenated segments, walked tile by tile with
// wave-uniform state: the segment, the keys it has left from the current
// tile on, and the byte address of the current tile's first key (segment base
// + the (b, h) offset + the rows already passed).  Total keys < 2^31 (checked
// on the host).
//
// FRAMED (fp8 K/V, one scale per frame): tiles never cross a frame.  A frame
// of F tokens is cut into ceil(F / 64) tiles, the last one partial when F is
// not a multiple of 64, and a segment's last frame may itself be partial; a
// segment starts on a frame boundary (frame-aligned arena spans).  frem holds
// the keys of the current frame from the current tile on.
template <bool FRAMED>
struct KeyStreamT {
  int s, rem, frem;
  int lim = 0x7FFFFFFF;  // keys past this index of the concatenated sequence are not part of the stream
  int b = 0;             // batch row, times each segment's batch stride (0: the head offset holds it)
  const char* ptr;
  __device__ __forceinline__ void enter(const void* const* base, int64_t head, const FlashParams& p, int seg) {
    s = seg;
    rem = (int)((p.seg_start[seg + 1] < lim ? p.seg_start[seg + 1] : (int64_t)lim) - p.seg_start[seg]);
    ptr = reinterpret_cast<const char*>(base[seg]) + (b * p.seg_bs[seg] + head);
    if constexpr (FRAMED) frem = p.frame;
  }
  __device__ __forceinline__ void seek(const void* const* base, int64_t head, int64_t tile_bytes,
                                       const FlashParams& p, int j) {
    int seg = 0;
    for (int i = 1; i < p.n_seg; ++i) seg = (j >= p.tile_start[i]) ? i : seg;
    enter(base, head, p, seg);
    const int t = j - p.tile_start[seg];
    if constexpr (FRAMED) {
      const int tpf = (p.frame + kBN - 1) / kBN;  // tiles per frame
      const int fr = t / tpf, k = t - fr * tpf;
      const int pos = fr * p.frame + k * kBN;
      frem = p.frame - k * kBN;
      rem -= pos;
      ptr += (int64_t)pos * (tile_bytes / kBN);
    } else {
      rem -= t * kBN;
      ptr += t * tile_bytes;
    }
  }
  __device__ __forceinline__ void next(const void* const* base, int64_t head, int64_t tile_bytes,
                                       const FlashParams& p) {
    if constexpr (FRAMED) {
      const int len = nvalid();
      rem -= len;
      ptr += (int64_t)len * (tile_bytes / kBN);
      frem -= len;
      if (frem == 0) frem = p.frame;
    } else {
      rem -= kBN;
      ptr += tile_bytes;
    }
    if (rem <= 0 && s + 1 < p.n_seg) enter(base, head, p, s + 1);
  }
  __device__ __forceinline__ int nvalid() const {
    const int n = rem < kBN ? rem : kBN;
    if constexpr (FRAMED) return frem < n ? frem : n;
    return n;
  }
  // first key of the current tile, counted from its segment's start
  __device__ __forceinline__ int row0(const FlashParams& p) const {
    return (int)(p.seg_start[s + 1] - p.seg_start[s]) - rem;
  }
};

// PAIR (both bodies below): 8-wave workgroups of two groups of 4 waves (waves
// w and w + 4 share a SIMD) that own two q-tiles of one head (pair_work) and
// read one K/V stream.  bf16: only group 0 issues the tile loads, so group
// 1's waves run their slot programs while group 0's wait on the load pipe.
// fp8: group 0 stages (loads and decodes) the K tiles and group 1 the V
// tiles, so each thread stages half of what a 4-wave workgroup's does for the
// same two q-tiles.  The groups meet at every per-tile barrier: the two
// waves of a SIMD finish together, where two 4-wave workgroups on one CU do
// not (the older one's waves win the issue arbitration and finish about a
// quarter earlier, leaving the CU half busy until the other ends).
template <int D, bool PAIR, bool VTOK>
__device__ __forceinline__ void flash_bf16_body(const FlashParams& p) {
  constexpr int BM = kBM, BN = kBN;
  constexpr int NKC = D / 8;         // 16-byte chunks of a K row
  constexpr int NVC = BN / 8;        // 16-byte chunks of a V^T row
  constexpr int KBUF = BN * D;       // elements of a K tile buffer
  constexpr int VBUF = D * BN;       // elements of a V^T tile buffer
  constexpr int KSLOT = KBUF / 512 / 4;  // load instructions (64 chunks) per wave and K tile
  constexpr int VSLOT = VBUF / 512 / 4;
  constexpr int CB = D / 16;         // 16-channel blocks of O
  constexpr int KS = D / 32;         // 32-channel steps of a score
  constexpr float kOver = 65536.0f;  // largest per-lane tile sum kept without raising m

  // K(0), K(1), V(0), V(1), one array: the output staging spans all four
  __shared__ __attribute__((aligned(16))) uint16_t smem[2 * (KBUF + VBUF)];
  uint16_t* const kbuf = smem;
  uint16_t* const vbuf = smem + 2 * KBUF;

  const int grp = PAIR ? (__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) >> 2) : 0;
  const WorkItem wi = PAIR ? pair_work(p, blockIdx.x, grp, p.tile_start[p.n_seg])
                           : work_item(p, blockIdx.x, p.tile_start[p.n_seg]);
  const bool loader = !PAIR || grp == 0;  // issues the K/V tile loads
  const int qt = wi.qtile % p.n_qtiles;
  const int bh = wi.qtile / p.n_qtiles;
  const int b = bh / p.H, h = bh % p.H;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) & 3;
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lg = lane >> 4;
  const int q0 = qt * BM + wave * 32 + li;  // this lane's queries: q0 and q0 + 16
  // a per-batch key count ends this row's key tiles early (the streams stop
  // at it, so its last tile is partial and masked like a segment's last)
  const int klim = p.n_klen ? p.klen[b] : 0x7FFFFFFF;
  int jend = wi.j1;
  if (p.n_klen) {
    const int tb = tiles_below(p, klim);
    jend = jend < tb ? jend : tb;
  }
  const int ntiles = jend > wi.j0 ? jend - wi.j0 : 0;

  // ---- per-lane load offsets (bytes from a tile's first key), loop invariant ----
  // Load slot i of wave w fills LDS chunks (w + 4 i) * 64 + lane.  The chunk's
  // row advances by 64 / chunks-per-row * 4 rows per slot, which leaves the
  // row's swizzle as it is, so the slots of a lane differ only by a uniform
  // number of keys (K) or channels (V): one offset per lane and operand.
  const int row_bytes = (int)(p.kv_ls * 2);
  const int vrow_bytes = (int)(p.v_ds * 2);
  const int krow0 = (wave * 64 + lane) / NKC, vrow0 = (wave * 64 + lane) / NVC;
  const int kchunk = (lane % NKC) ^ row_swizzle<NKC>(krow0);
  const int vchunk = VTOK ? (lane % NKC) ^ key_swizzle<NKC>(krow0) : (lane % NVC) ^ row_swizzle<NVC>(vrow0);
  const int koff = key_of_row(krow0) * row_bytes + kchunk * 16;
  const int voff = (VTOK ? krow0 * row_bytes : vrow0 * vrow_bytes) + vchunk * 16;
  auto kslot_keys = [](int i) { return key_of_row(i * (256 / NKC)); };  // keys from slot 0's to slot i's

  const int64_t k_head = h * p.kv_hs * 2;
  const int64_t v_head = VTOK ? k_head : (b * p.v_bs + h * p.v_hs) * 2;
  const int64_t k_tile = (int64_t)BN * row_bytes;
  const int64_t v_tile = VTOK ? k_tile : BN * 2;
  KeyStreamT<false> kit, vit;
  kit.lim = klim;
  vit.lim = klim;
  kit.b = b;
  vit.b = VTOK ? b : 0;
  kit.seek(p.k_ptr, k_head, k_tile, p, wi.j0);
  vit.seek(p.v_ptr, v_head, v_tile, p, wi.j0);
  // LDS address of this wave's first load slot in a buffer; the empty asm
  // keeps the compiler from holding every (buffer, slot) address in its own
  // scalar register across the loop (they cost one s_add each instead)
  auto lds_slot0 = [&](uint16_t* buf0) {
    uint32_t a = (uint32_t)(uintptr_t)(lds_ptr_t)(buf0 + wave * 512);
    asm volatile("" : "+s"(a));
    return a;
  };
  // The tile's loads.  K rows past a segment's end lie outside the partial
  // tile's buffer range (a whole tile's is left open): those lanes load
  // zeros, and their scores are masked out of the softmax.  A whole tile's
  // slots take their uniform offset from a scalar register; a partial tile
  // adds it per lane, so the range check sees the whole offset.  Token-major V
  // is bounded the same way; key-major V (8-key chunks of its rows) re-reads
  // the segment's last chunk for the positions past its end.
  auto issue_k = [&](int buf) {
    const int nv = kit.nvalid();
    const uint32_t l0 = lds_slot0(kbuf + buf * KBUF);
    if (loader) {
      if (nv == BN) {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)kit.ptr, (short)0, 0x7FFFFFFF, 0x00020000);
#pragma unroll
        for (int i = 0; i < KSLOT; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(uintptr_t)(l0 + i * 4096), 16, koff,
                                                   kslot_keys(i) * row_bytes, 0, 0);
      } else {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)kit.ptr, (short)0, nv * row_bytes, 0x00020000);
#pragma unroll
        for (int i = 0; i < KSLOT; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(uintptr_t)(l0 + i * 4096), 16,
                                                   koff + kslot_keys(i) * row_bytes, 0, 0, 0);
      }
    }
    kit.next(p.k_ptr, k_head, k_tile, p);
  };
  auto issue_v = [&](int buf) {
    const uint32_t l0 = lds_slot0(vbuf + buf * VBUF);
    const int nv = vit.nvalid();
    if (VTOK && loader) {
      const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)vit.ptr, (short)0,
                                                        nv == BN ? 0x7FFFFFFF : nv * row_bytes, 0x00020000);
      const bool whole = nv == BN;
#pragma unroll
      for (int i = 0; i < VSLOT; ++i) {
        const int step = i * (256 / NKC) * row_bytes;
        if (whole)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(uintptr_t)(l0 + i * 4096), 16, voff, step, 0, 0);
        else
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(uintptr_t)(l0 + i * 4096), 16, voff + step, 0, 0,
                                                   0);
      }
    }
    if (!VTOK && loader) {
      const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)vit.ptr, (short)0, 0x7FFFFFFF, 0x00020000);
      int off = voff;
      if (nv < BN) off = vrow0 * vrow_bytes + min(vchunk, (nv + 7) / 8 - 1) * 16;
#pragma unroll
      for (int i = 0; i < VSLOT; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(uintptr_t)(l0 + i * 4096), 16, off,
                                                 i * (256 / NVC) * vrow_bytes, 0, 0);
    }
    vit.next(p.v_ptr, v_head, v_tile, p);
  };

  // ---- Q^T fragments, resident for the whole key loop ----
  bf16x8_t qf[2][KS];
  auto load_q = [&]() {
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int qi = q0 + 16 * n;
      const bool ok = qi < p.Lq;
      const uint16_t* qp = p.q + b * p.q_bs + (int64_t)(ok ? qi : 0) * p.q_ls + h * p.q_hs + lg * 8;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const uint4 v = ok ? *reinterpret_cast<const uint4*>(qp + s * 32) : make_uint4(0, 0, 0, 0);
        qf[n][s] = __builtin_bit_cast(bf16x8_t, v);
      }
    }
  };

  f32x4_t oacc[CB][2];
#pragma unroll
  for (int d = 0; d < CB; ++d) oacc[d][0] = oacc[d][1] = f32x4_t{};
  const float c = p.scale_log2;  // > 0
  float m_run[2] = {-INFINITY, -INFINITY};  // per query, base-2 logit units
  float l_run[2] = {0.0f, 0.0f};            // this lane's share of the row sums
  const ltx_bf16x2_t ones = __builtin_bit_cast(ltx_bf16x2_t, 0x3F803F80u);  // bf16 pair (1, 1)

  // Scores: s[kb][n][r] is query q0 + 16 n over key 32 (kb / 2) + 8 lg + 4 (kb % 2) + r
  // of the tile; score pair q (two adjacent r) of the softmax and of P is
  // kb = 2 (q / 8) + (q % 4) / 2, n = (q / 4) % 2, r = 2 (q % 2) + {0, 1},
  // so P words 8 k2 + 4 n .. + 3 are the B operand of key half k2.
  // keys past a partial tile's valid count drop out of the softmax (compare
  // the key's constant part with one per-lane limit)
  auto mask_tail = [&](f32x4_t (&s)[4][2], int nvalid) {
    const int lim = nvalid - 8 * lg;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (32 * (kb >> 1) + 4 * (kb & 1) + r >= lim) s[kb][0][r] = s[kb][1][r] = -INFINITY;
  };
  // largest base-2 logit of a tile for this lane's query n
  auto tile_max = [&](const f32x4_t (&s)[4][2], int n) {
    float mt = s[0][n][0];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) mt = fmaxf(mt, s[kb][n][r]);
    return quad_max(mt) * c;
  };
  // P = 2^(S*c + neg_m) of query n packed to bf16 pairs; returns this lane's
  // sum of the packed values.  Used outside the slot program (first tile,
  // rescale), where one key may dominate: the sum of the rounded P then
  // cancels its rounding in O.
  auto exp_all = [&](const f32x4_t (&s)[4][2], uint32_t (&pw)[16], int n, float neg_m) {
    float ps = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int q = (i >> 2) * 8 + n * 4 + (i & 3), kb = 2 * (q >> 3) + ((q & 3) >> 1), r = 2 * (q & 1);
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][n][r], c, neg_m));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][n][r + 1], c, neg_m));
      pw[q] = pack_bf16x2(p0, p1);
      ps = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(ltx_bf16x2_t, pw[q]), ones, ps, false);
    }
    return ps;
  };
  // Fragments: lane (li, lg) reads row li of a 16-row block, 16-byte chunk
  // 4 * step + lg, stored at the chunk index xor the row's swizzle.  The
  // blocks' row offsets are multiples of 16 rows and a step only flips offset
  // bits (4 chunks = 32 elements), so one offset per operand serves every
  // fragment.
  const int kofs = li * D + (lg ^ row_swizzle<NKC>(li)) * 8;
  const int vofs = li * BN + (lg ^ row_swizzle<NVC>(li)) * 8;
  auto kfrag = [&](int buf, int kb, int s) -> bf16x8_t {
    return *reinterpret_cast<const bf16x8_t*>(kbuf + buf * KBUF + kb * 16 * D + (kofs ^ (s * 32)));
  };
  // Token-major V tiles hold keys in rows, so a V^T fragment is read with the
  // transposing LDS read: the 16 lanes of one lg read a block of 4 keys x 16
  // channels (8 bytes per lane) and lane li receives its channel of the 4
  // keys; two reads give the lane's 8 keys.
  const int tofs = (8 * lg + (li >> 2)) * D + (((li >> 1) & 1) ^ key_swizzle<NKC>(8 * lg + (li >> 2))) * 8 +
                   (li & 1) * 4;
  auto vfrag = [&](int buf, int d, int k2) -> bf16x8_t {
    if constexpr (VTOK) {
      typedef short s16x4_t __attribute__((ext_vector_type(4)));
      typedef short s16x8_t __attribute__((ext_vector_type(8)));
      typedef __attribute__((address_space(3))) s16x4_t* lds_s16x4_t;
      uint16_t* v0 = vbuf + buf * VBUF + 32 * k2 * D + (tofs ^ (16 * d));
      const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)v0);
      const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(v0 + 4 * D));
      return __builtin_bit_cast(bf16x8_t, (s16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      return *reinterpret_cast<const bf16x8_t*>(vbuf + buf * VBUF + d * 16 * BN + (vofs ^ (k2 * 32)));
    }
  };
  auto pfrag = [](const uint32_t (&pw)[16], int k2, int n) {
    const int q = 8 * k2 + 4 * n;
    return __builtin_bit_cast(bf16x8_t, make_uint4(pw[q], pw[q + 1], pw[q + 2], pw[q + 3]));
  };
  // S = K Q^T of a whole tile (first tiles only)
  auto qk_tile = [&](int buf, f32x4_t (&s)[4][2]) {
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const bf16x8_t a = kfrag(buf, kb, k);
#pragma unroll
        for (int n = 0; n < 2; ++n)
          s[kb][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[n][k], k == 0 ? f32x4_t{} : s[kb][n], 0, 0, 0);
      }
  };
  // O^T += V^T P^T of a whole tile (last tile only)
  auto pv_tile = [&](int buf, const uint32_t (&pw)[16]) {
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
      for (int d = 0; d < CB; ++d) {
        const bf16x8_t a = vfrag(buf, d, k2);
#pragma unroll
        for (int n = 0; n < 2; ++n)
          oacc[d][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pfrag(pw, k2, n), oacc[d][n], 0, 0, 0);
      }
  };
  // the tile loads go straight to LDS and are counted by vmcnt, so they must
  // land before the barrier publishes them
  auto publish = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };

  // ---- the slot program of one tile ----
  // NS slots: PV(j-1) (2*CB fragments of V(j-1)) then S(j+1) (4*KS fragments
  // of K(j+1)).  Each slot issues the two MFMAs of its fragment (the lane's
  // two queries), the LDS read of the fragment PREF slots ahead, and a slice
  // of the softmax of S(j).  With 32 slots (D = 128) that is one score per
  // slot: score i has its fma at slot i, its exp at i + 1 and its row-sum add
  // at i + 2, and pair q its bf16 pack at 2q + 3 (whole pairs per slot, fma
  // of both at 2q and the rest at 2q + 1 and 2q + 3, measured 1 % slower: the
  // odd slots then carry two exps, the adds and the pack).  With 16 slots
  // (D = 64) score pair p has its fma at slot p, its exp at p + 1 and its
  // pack and adds at p + 3.  A scheduling fence closes every slot, so the exp
  // work stays spread under the MFMAs.  The row sum adds the fp32 P
  // values: v_dot2c_f32_bf16 over the packed pair (one instruction instead
  // of two) waits for the SIMD's matrix pipeline on gfx950, about one MFMA
  // per instruction while the other wave's MFMAs run, where adds issue
  // beside them.
  constexpr int NPV = 2 * CB, NS = NPV + 4 * KS;
  constexpr int PREF = 3;
  auto tile = [&](int vb, int kbf, const f32x4_t (&scur)[4][2], f32x4_t (&snext)[4][2], const uint32_t (&pprev)[16],
                  uint32_t (&pcur)[16], float (&ps)[2], const float (&neg_m)[2], auto&& loads) {
    auto frag = [&](int t) -> bf16x8_t {
      if (t < NPV) return vfrag(vb, t % CB, t / CB);
      return kfrag(kbf, (t - NPV) & 3, (t - NPV) >> 2);
    };
    bf16x8_t ring[PREF + 1];
#pragma unroll
    for (int t = 0; t < PREF; ++t) ring[t] = frag(t);
    float e0[16], e1[16];
    ps[0] = ps[1] = 0.0f;
#pragma unroll
    for (int t = 0; t < NS + 2; ++t) {
      if (t < NS) {
        if (t + PREF < NS) ring[(t + PREF) % (PREF + 1)] = frag(t + PREF);
        const bf16x8_t a = ring[t % (PREF + 1)];
        if (VTOK && t == NPV - PREF) loads();
        // the query blocks alternate (0 1, 1 0, ...): consecutive MFMAs share an operand
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int n = i ^ (t & 1);
          if (t < NPV) {
            oacc[t % CB][n] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pfrag(pprev, t / CB, n), oacc[t % CB][n], 0, 0, 0);
          } else {
            const int kb = (t - NPV) & 3, kk = (t - NPV) >> 2;  // the four key blocks' chains alternate
            snext[kb][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[n][kk], kk == 0 ? f32x4_t{} : snext[kb][n],
                                                                   0, 0, 0);
          }
        }
      }
      if constexpr (NS == 32) {
        // one score per slot: its fma at slot i, its exp at i + 1, its
        // row-sum add at i + 2, and the bf16 pack of pair q at 2q + 3, so
        // every slot carries the same vector work
#pragma unroll
        for (int i = 0; i < 32; ++i) {
          const int q = i >> 1, n = (q >> 2) & 1, kb = 2 * (q >> 3) + ((q & 3) >> 1), r = 2 * (q & 1) + (i & 1);
          float* e = (i & 1) ? e1 : e0;
          if (t == i) e[q] = __builtin_fmaf(scur[kb][n][r], c, neg_m[n]);
          if (t == i + 1) e[q] = __builtin_amdgcn_exp2f(e[q]);
          if (t == i + 2) ps[n] = ps[n] + e[q];
        }
#pragma unroll
        for (int q = 0; q < 16; ++q)
          if (t == 2 * q + 3) {
            pcur[q] = pack_bf16x2(e0[q], e1[q]);
            // with no use left in this slot the compiler would sink the pack
            // to the next tile's PV and issue all sixteen back to back after
            // the slot program; pin it here, under this slot's MFMAs
            asm volatile("" : "+v"(pcur[q]));
          }
      } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int n = (q >> 2) & 1, kb = 2 * (q >> 3) + ((q & 3) >> 1), r = 2 * (q & 1);
          if ((2 * q * NS) / 32 == t) {
            e0[q] = __builtin_fmaf(scur[kb][n][r], c, neg_m[n]);
            e1[q] = __builtin_fmaf(scur[kb][n][r + 1], c, neg_m[n]);
          }
          if ((2 * q * NS) / 32 + 1 == t) {
            e0[q] = __builtin_amdgcn_exp2f(e0[q]);
            e1[q] = __builtin_amdgcn_exp2f(e1[q]);
          }
          if ((2 * q * NS) / 32 + 3 == t || (q == 15 && t == NS + 1 && (2 * q * NS) / 32 + 3 > NS + 1)) {
            pcur[q] = pack_bf16x2(e0[q], e1[q]);
            ps[n] = ps[n] + e0[q];
            ps[n] = ps[n] + e1[q];
            asm volatile("" : "+v"(pcur[q]));
          }
        }
      }
      // the slot's order: MFMA, exp, MFMA, fragment read, other vector work
      // (144 us at 1152 x 4608 against 145 us in the compiler's order and
      // 147-149 us with both MFMAs first)
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      if (VTOK && t + PREF < NPV)
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      else
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  if (ntiles > 0) {
    f32x4_t sa[4][2], sb[4][2];
    uint32_t pa[16], pb[16];  // P(j) of even / odd j
    // ---- prologue: S(0) sets m from its own maximum; P(0); S(1) ----
    issue_k(0);
    if (ntiles > 1) issue_k(1);
    const int nv0 = vit.nvalid();  // valid keys of tile 0 (the V stream is at tile j before V(j) is issued)
    issue_v(0);
    load_q();  // its latency overlaps the first tiles' loads
    publish();
    qk_tile(0, sa);
    if (nv0 < BN) mask_tail(sa, nv0);
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      m_run[n] = tile_max(sa, n);
      l_run[n] = exp_all(sa, pa, n, -m_run[n]);
    }
    if (ntiles > 1) qk_tile(1, sb);
    if (ntiles > 2) {
      __syncthreads();  // every wave is done with K(0)
      issue_k(0);       // K(2)
    }
    // ---- iteration j (1 <= j < ntiles), of parity jp: the slot program
    //      computes O += V(j-1)^T P(j-1), S(j+1) = K(j+1) Q^T and
    //      P(j) = 2^(S(j)c - m).  On the last tile S(j+1) is computed from
    //      stale LDS and dropped. ----
    auto step = [&](int j, auto jpar, f32x4_t (&scur)[4][2], f32x4_t (&snext)[4][2], const uint32_t (&pprev)[16],
                    uint32_t (&pcur)[16]) {
      constexpr int jp = decltype(jpar)::value;
      publish();  // K(j+1) and V(j-1) have landed; the buffers of K(j) and V(j-2) are free
      const int nv = vit.nvalid();  // valid keys of tile j
      auto loads = [&]() {
        if (j + 2 < ntiles) issue_k(jp);  // K(j+2)
        issue_v(jp);                      // V(j)
      };
      // Token-major V: after the tile's last V fragment read instead (the
      // compiler waits for every load to LDS in flight before a transposing
      // read: 178 us with the loads here, at 1152 x 4608).
      if (!VTOK) loads();
      if (nv < BN) mask_tail(scur, nv);
      const float neg_m[2] = {-m_run[0], -m_run[1]};
      float ps[2];
      tile(1 - jp, 1 - jp, scur, snext, pprev, pcur, ps, neg_m, loads);
      if (__builtin_amdgcn_ballot_w64(fmaxf(ps[0], ps[1]) > kOver)) {
        // raise m to the tile maximum, rescale O and l, redo P(j) from S(j)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          const float m_new = fmaxf(m_run[n], tile_max(scur, n));
          const float alpha = __builtin_amdgcn_exp2f(m_run[n] - m_new);
          m_run[n] = m_new;
          l_run[n] *= alpha;
#pragma unroll
          for (int d = 0; d < CB; ++d) oacc[d][n] *= alpha;
          ps[n] = exp_all(scur, pcur, n, -m_run[n]);
        }
      }
      l_run[0] += ps[0];
      l_run[1] += ps[1];
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    int j = 1;
    for (; j + 1 < ntiles; j += 2) {
      step(j, odd, sb, sa, pa, pb);
      step(j + 1, even, sa, sb, pb, pa);
    }
    if (j < ntiles) step(j, odd, sb, sa, pa, pb);
    // ---- epilogue: O += V(n-1)^T P(n-1) ----
    publish();
    if ((ntiles - 1) & 1)
      pv_tile(1, pb);
    else
      pv_tile(0, pa);
  }

  // output staging: 32 rows of D per wave
  static_assert((PAIR ? 8 : 4) * 32 * D <= 2 * (KBUF + VBUF), "output staging region");
  const int owave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const float l_tot[2] = {quad_sum(l_run[0]), quad_sum(l_run[1])};
  finish_rows<D, stores_f32_partials(D, PAIR, VTOK)>(p, wi, b, h, qt, wave * 32, oacc, m_run, l_tot, smem + owave * 32 * D);
}

// The 32x32x16 body: the fp8 kernels, and bf16 key-major V where the part is
// not power bound (small_grid).  FRAMED (fp8 only): frames that are not a whole
// number of 64-key tiles, cut at frame boundaries (KeyStreamT<true>, its own
// kernel); frames of 64k tokens take the plain tiling, which never crosses a
// frame either and keeps the hot kernel's scalar state and registers as they
// were (the framed state costs the D = 128 instance register spills).
template <int D, bool FP8, bool FRAMED, bool PAIR = false>
__device__ __forceinline__ void flash_mfma32_body(const FlashParams& p) {
  static_assert(FP8 || !FRAMED, "frame tiling is an fp8 feature");
  static_assert(!PAIR || (FP8 && !FRAMED), "pair workgroups: fp8 in the plain tiling");
  constexpr int BM = kBM, BN = kBN;
  constexpr int NKC = D / 8;
  constexpr int KS = D + 8;
  // V^T tile rows (one head-dim channel, BN keys = 8 chunks of 16 bytes):
  // with D = 128 two rows share one pad chunk (17 chunks per pair, 17 load
  // instructions per tile), else each row has its own (9 chunks).  Either
  // way 16 consecutive rows' same chunk covers 16 distinct 16-byte bank
  // groups, so a fragment read is conflict-free.
  constexpr bool VPAIR = (D / 2) * 17 % 64 == 0;
  constexpr int VS = BN + 8;                      // row stride without pairing
  constexpr int VPS = 2 * BN + 8;                 // pair stride with pairing
  constexpr int KBUF = BN * KS;
  constexpr int VBUF = VPAIR ? (D / 2) * VPS : D * VS;
  constexpr int KINS = BN * (NKC + 1) / 64;
  constexpr int VINS = VPAIR ? (D / 2) * 17 / 64 : D * 9 / 64;
  constexpr int KSLOT = (KINS + 3) / 4;
  constexpr int VSLOT = (VINS + 3) / 4;
  constexpr int DB = D / 32;
  constexpr int QS = D / 16;
  constexpr float kOver = 65536.0f;  // largest per-lane tile sum kept without raising m
  static_assert(BN * (NKC + 1) % 64 == 0 && (VPAIR || D * 9 % 64 == 0), "tile does not split into whole instructions");
  // element offset of V^T row r in a V buffer
  auto vrow = [](int r) { return VPAIR ? (r >> 1) * VPS + (r & 1) * BN : r * VS; };

  __shared__ __attribute__((aligned(16))) uint16_t kbuf[2][KBUF];
  __shared__ __attribute__((aligned(16))) uint16_t vbuf[2][VBUF];

  const int grp = PAIR ? (__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) >> 2) : 0;
  const WorkItem wi = PAIR ? pair_work(p, blockIdx.x, grp, p.tile_start[p.n_seg])
                           : work_item(p, blockIdx.x, p.tile_start[p.n_seg]);
  const int qt = wi.qtile % p.n_qtiles;
  const int bh = wi.qtile / p.n_qtiles;
  const int b = bh / p.H, h = bh % p.H;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) & 3;
  const int lane = threadIdx.x & 63;
  const int li = lane & 31, hg = lane >> 5;
  const int qi = qt * BM + wave * 32 + li;
  // a per-batch key count ends this row's key tiles early (the streams stop
  // at it, so its last tile is partial and masked like a segment's last)
  const int klim = (!FP8 && p.n_klen) ? p.klen[b] : 0x7FFFFFFF;
  int jend = wi.j1;
  if (!FP8 && p.n_klen) {
    const int tb = tiles_below(p, klim);
    jend = jend < tb ? jend : tb;
  }
  const int ntiles = jend > wi.j0 ? jend - wi.j0 : 0;

  // ---- per-lane load offsets (bytes from a tile's first key), loop invariant ----
  const int row_bytes = (int)(p.kv_ls * (FP8 ? 1 : 2));
  const int vrow_bytes = (int)(p.v_ds * 2);
  auto kpos = [&](int i, int& r, int& c) {
    const int pch = (wave + 4 * i) * 64 + lane;
    r = sig(pch / (NKC + 1));
    c = pch % (NKC + 1);
    c = c < NKC ? c : 0;
  };
  // the (channel, 16-byte chunk) load slot i of this lane fills; a pad slot
  // re-reads a valid chunk
  auto vpos = [&](int i, int& d, int& c) {
    const int pch = (wave + 4 * i) * 64 + lane;
    if constexpr (VPAIR) {
      const int q = pch % 17;
      d = 2 * (pch / 17) + (q < 16 ? q >> 3 : 0);
      c = q < 16 ? (q & 7) : 0;
    } else {
      d = pch / 9;
      d = d < D ? d : 0;
      c = pch % 9;
      c = c < 8 ? c : 0;
    }
  };
  int koff[KSLOT], voff[VSLOT];
#pragma unroll
  for (int i = 0; i < KSLOT; ++i) {
    int r, c;
    kpos(i, r, c);
    koff[i] = r * row_bytes + c * 16;
  }
#pragma unroll
  for (int i = 0; i < VSLOT; ++i) {
    int d, c;
    vpos(i, d, c);
    voff[i] = d * vrow_bytes + c * 16;
  }

  const int64_t k_head = h * p.kv_hs * (FP8 ? 1 : 2);
  const int64_t v_head = FP8 ? k_head : (b * p.v_bs + h * p.v_hs) * 2;
  const int64_t k_tile = (int64_t)BN * row_bytes;
  const int64_t v_tile = FP8 ? k_tile : BN * 2;
  KeyStreamT<FRAMED> kit, vit;
  kit.lim = klim;
  vit.lim = klim;
  kit.b = b;
  vit.b = FP8 ? b : 0;
  kit.seek(p.k_ptr, k_head, k_tile, p, wi.j0);
  vit.seek(p.v_ptr, v_head, v_tile, p, wi.j0);
  // LDS address of this wave's first load slot in a buffer; the empty asm
  // keeps the compiler from holding every (buffer, slot) address in its own
  // scalar register across the loop (they cost one s_add each instead)
  auto lds_slot0 = [&](uint16_t* buf0) {
    uint32_t a = (uint32_t)(uintptr_t)(lds_ptr_t)(buf0 + wave * 512);
    asm volatile("" : "+s"(a));
    return a;
  };
  // One load instruction ("slot" i of this wave) of a K or V tile.  rs is the
  // tile's buffer resource, l0 this wave's first LDS chunk of the buffer and
  // nv the tile's valid keys.  K rows past a segment's end lie outside the
  // partial tile's buffer range (issue_k): those lanes load zeros, and their
  // scores are masked out of the softmax.  V (8-key chunks of key-major rows)
  // re-reads the segment's last chunk for the positions past its end.
  auto k_load = [&](__amdgpu_buffer_rsrc_t rs, uint32_t l0, int i) {
    if (i < KSLOT && wave + 4 * i < KINS)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(uintptr_t)(l0 + i * 4096), 16, koff[i], 0, 0, 0);
  };
  auto v_load = [&](__amdgpu_buffer_rsrc_t rs, uint32_t l0, int nv, int i) {
    if (i < VSLOT && wave + 4 * i < VINS) {
      int off = voff[i];
      if (nv < BN) {
        int d, c;
        vpos(i, d, c);
        off = d * vrow_bytes + min(c, (nv + 7) / 8 - 1) * 16;
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(uintptr_t)(l0 + i * 4096), 16, off, 0, 0, 0);
    }
  };
  auto rsrc = [&](const char* ptr) { return __builtin_amdgcn_make_buffer_rsrc((void*)ptr, (short)0, 0x7FFFFFFF, 0x00020000); };
  // whole tiles (every tile but a segment's last) take one branch and issue
  // their loads from the precomputed offsets; a K tile's buffer range ends at
  // its last valid row (a whole tile's is left open), so the partial tile
  // issues the same loads
  auto issue_k = [&](int buf) {
    const int nv = kit.nvalid();
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)kit.ptr, (short)0, nv == BN ? 0x7FFFFFFF : nv * row_bytes,
                                                      0x00020000);
    const uint32_t l0 = lds_slot0(kbuf[buf]);
#pragma unroll
    for (int i = 0; i < KSLOT; ++i) k_load(rs, l0, i);
    kit.next(p.k_ptr, k_head, k_tile, p);
  };
  auto issue_v = [&](int buf) {
    const auto rs = rsrc(vit.ptr);
    const uint32_t l0 = lds_slot0(vbuf[buf]);
    const int nv = vit.nvalid();
    if (nv == BN) {
#pragma unroll
      for (int i = 0; i < VSLOT; ++i) v_load(rs, l0, BN, i);
    } else {
#pragma unroll
      for (int i = 0; i < VSLOT; ++i) v_load(rs, l0, nv, i);
    }
    vit.next(p.v_ptr, v_head, v_tile, p);
  };

  // ---- fp8: register staging of the next K and V tiles ----
  // K: thread t moves 8-code chunk t % NKC of rows t / NKC + FROWS * i.
  // V: thread t (< NVP) moves 8-channel chunk t / 16 of keys 4 * (t % 16) .. +3
  // and writes them transposed (4 keys of 8 channel rows); 16 consecutive
  // lanes fill one 128-byte V^T row segment, so the LDS writes are
  // conflict-free.  Loads past a partial tile's last key return 0 (buffer
  // range check).
  constexpr int FROWS = 256 / NKC;
  constexpr int FKL = BN / FROWS;
  constexpr int NVP = (BN / 4) * NKC;
  const int tid = threadIdx.x & 255;  // thread index within the group
  const int fkc = tid % NKC, fkr = tid / NKC;
  const int fvg = tid % 16, fvc = tid / 16;
  const bool fv_on = tid < NVP;
  const bool stage_k = !PAIR || grp == 0, stage_v = !PAIR || grp == 1;  // wave-uniform
  uint2 kreg[FP8 ? FKL : 1], vreg[FP8 ? 4 : 1];
  auto load_k8 = [&]() {
    if (!stage_k) return;
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)kit.ptr, (short)0, kit.nvalid() * row_bytes, 0x00020000);
#pragma unroll
    for (int i = 0; i < FKL; ++i) kreg[i] = KVChunk<true>::bload(rs, (fkr + FROWS * i) * row_bytes + fkc * 8);
    kit.next(p.k_ptr, k_head, k_tile, p);
  };
  auto load_v8 = [&]() {
    if (!stage_v) return;
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)vit.ptr, (short)0, vit.nvalid() * row_bytes, 0x00020000);
    if (fv_on) {
#pragma unroll
      for (int e = 0; e < 4; ++e) vreg[e] = KVChunk<true>::bload(rs, (fvg * 4 + e) * row_bytes + fvc * 8);
    }
    vit.next(p.v_ptr, v_head, v_tile, p);
  };
  auto store_k8_row = [&](int buf, int i) {
    if (!stage_k) return;
    *reinterpret_cast<uint4*>(&kbuf[buf][sig(fkr + FROWS * i) * KS + fkc * 8]) = KVChunk<true>::to_bf16(kreg[i]);
  };
  auto store_k8 = [&](int buf) {
#pragma unroll
    for (int i = 0; i < FKL; ++i) store_k8_row(buf, i);
  };
  auto store_v8_half = [&](int buf, int half) {
    if constexpr (FP8) {   // vreg holds the four staged code chunks only in the fp8 instances
      if (!stage_v || !fv_on) return;
      const uint32_t d0 = half ? vreg[0].y : vreg[0].x, d1 = half ? vreg[1].y : vreg[1].x;
      const uint32_t d2 = half ? vreg[2].y : vreg[2].x, d3 = half ? vreg[3].y : vreg[3].x;
      // channels 4*half + {0, 1} and {2, 3} of keys (0, 1) and (2, 3)
      const uint32_t k01a = __builtin_amdgcn_perm(d1, d0, 0x05010400u), k23a = __builtin_amdgcn_perm(d3, d2, 0x05010400u);
      const uint32_t k01b = __builtin_amdgcn_perm(d1, d0, 0x07030602u), k23b = __builtin_amdgcn_perm(d3, d2, 0x07030602u);
      const int r0 = fvc * 8 + 4 * half;
      uint16_t* vb = &vbuf[buf][fvg * 4];
      *reinterpret_cast<uint2*>(vb + vrow(r0)) = make_uint2(KVChunk<true>::pair(k01a, false), KVChunk<true>::pair(k23a, false));
      *reinterpret_cast<uint2*>(vb + vrow(r0 + 1)) = make_uint2(KVChunk<true>::pair(k01a, true), KVChunk<true>::pair(k23a, true));
      *reinterpret_cast<uint2*>(vb + vrow(r0 + 2)) = make_uint2(KVChunk<true>::pair(k01b, false), KVChunk<true>::pair(k23b, false));
      *reinterpret_cast<uint2*>(vb + vrow(r0 + 3)) = make_uint2(KVChunk<true>::pair(k01b, true), KVChunk<true>::pair(k23b, true));
    }
  };
  // V(j) to LDS: the codes are interleaved by key before decoding: one v_perm
  // puts channels c and c + 1 of keys 2i and 2i + 1 into one word, whose low
  // and high byte pairs decode into the (key 2i, key 2i + 1) bf16 pairs of the
  // two V^T rows.  8 perms and 16 decodes per thread, where decoding first and
  // transposing the bf16 pairs takes 16 of each.
  auto store_v8 = [&](int buf) {
    store_v8_half(buf, 0);
    store_v8_half(buf, 1);
  };
  // the tile the softmax works on: its valid keys and (fp8) its scales
  KeyStreamT<FRAMED> cit;
  if constexpr (FP8) cit.seek(p.k_ptr, 0, 0, p, wi.j0);
  struct TileScale { float c, off, inv; };  // logit scale, exponent offset log2 sv, 1 / sv
  auto tile_scale = [&]() -> TileScale {
    if constexpr (FP8) {
      const int64_t o = b * p.sc_bs + h * p.sc_hs + cit.row0(p) / p.frame;
      const float sk = p.k_sc[cit.s][o];
      const float sv = p.v_sc[cit.s][o];
      return TileScale{p.scale_log2 * sk, __log2f(sv), 1.0f / sv};
    } else {
      return TileScale{p.scale_log2, 0.0f, 1.0f};
    }
  };

  // ---- Q^T fragments, resident for the whole key loop ----
  bf16x8_t qf[QS];
  auto load_q = [&]() {
    const bool ok = qi < p.Lq;
    const uint16_t* qp = p.q + b * p.q_bs + (int64_t)(ok ? qi : 0) * p.q_ls + h * p.q_hs + hg * 8;
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      uint4 v = ok ? *reinterpret_cast<const uint4*>(qp + s * 16) : make_uint4(0, 0, 0, 0);
      qf[s] = __builtin_bit_cast(bf16x8_t, v);
    }
  };

  f32x16_t oacc[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d) oacc[d] = f32x16_t{};
  float m_run = -INFINITY;  // per query, base-2 logit units
  float l_run = 0.0f;       // this lane's share of the row sum
  const ltx_bf16x2_t ones = __builtin_bit_cast(ltx_bf16x2_t, 0x3F803F80u);  // bf16 pair (1, 1)

  // keys past a partial tile's valid count drop out of the softmax (the
  // lane's key is kb*32 + 16*(r/8) + 8*hg + r%8: compare its constant part
  // with one per-lane limit so no key index is kept in registers)
  auto mask_tail = [&](f32x16_t (&s)[2], int nvalid) {
    const int lim = nvalid - 8 * hg;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (kb * 32 + 16 * (r >> 3) + (r & 7) >= lim) s[kb][r] = -INFINITY;
  };
  // largest base-2 logit of a tile for this lane's query (c > 0)
  auto tile_max = [&](const f32x16_t (&s)[2], float c) {
    float mt = s[0][0];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[kb][r]);
    return pair_max(mt) * c;
  };
  // P = 2^(S*c + off) packed to bf16 pairs (pw[i] holds scores 2i, 2i+1 in
  // accumulator order); returns this lane's sum.  Used outside the slot
  // program (first tile, rescale).
  auto exp_all = [&](const f32x16_t (&s)[2], uint32_t (&pw)[16], float c, float neg_m) {
    float ps = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; i += 2) {
      const int kb = i >> 4, r = i & 15;
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r], c, neg_m));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r + 1], c, neg_m));
      pw[i >> 1] = pack_bf16x2(p0, p1);
      ps = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(ltx_bf16x2_t, pw[i >> 1]), ones, ps, false);
    }
    return ps;
  };
  // S = K Q^T of a whole tile from kbuf[buf] (first tile only)
  auto qk_tile = [&](int buf, f32x16_t (&s)[2]) {
    const f32x16_t zero = f32x16_t{};
    const uint16_t* kf = &kbuf[buf][li * KS + hg * 8];
#pragma unroll
    for (int k = 0; k < QS; ++k) {
      const bf16x8_t a0 = *reinterpret_cast<const bf16x8_t*>(kf + k * 16);
      const bf16x8_t a1 = *reinterpret_cast<const bf16x8_t*>(kf + 32 * KS + k * 16);
      s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, qf[k], k == 0 ? zero : s[0], 0, 0, 0);
      s[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, qf[k], k == 0 ? zero : s[1], 0, 0, 0);
    }
  };
  // O^T += V^T P^T of a whole tile from vbuf[buf] (last tile only)
  auto pv_tile = [&](int buf, const uint32_t (&pw)[16]) {
    const uint16_t* vf = &vbuf[buf][vrow(li) + hg * 8];
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
      const bf16x8_t pf =
          __builtin_bit_cast(bf16x8_t, make_uint4(pw[4 * k4], pw[4 * k4 + 1], pw[4 * k4 + 2], pw[4 * k4 + 3]));
#pragma unroll
      for (int d = 0; d < DB; ++d)
        oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            *reinterpret_cast<const bf16x8_t*>(vf + vrow(d * 32) + k4 * 16), pf, oacc[d], 0, 0, 0);
    }
  };
  // bf16: the tile loads go straight to LDS and are counted by vmcnt, so
  // they must land before the barrier publishes them.  fp8: the staged tiles
  // reach LDS through ds_writes (the barrier waits for those), and the
  // loads in flight only fill registers that the next slot program decodes
  // (the compiler waits for each before its use), so they stay in flight
  // across the barrier: 194.5 -> 192.8 us at 1152 x 4608.
  auto publish = [&]() {
    if constexpr (!FP8) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };

  // ---- the slot program of one tile ----
  // NS matrix-core slots: PV(j-1) (4*DB MFMAs over vbuf[vb]) then S(j+1)
  // (2*QS MFMAs over kbuf[kbf]).  Each slot issues its MFMA, the LDS read
  // of the fragment PREF slots ahead, and a slice of the softmax of S(j).
  // With 32 slots (D = 128) that is one score per slot: score i has its fma
  // at slot i, its exp at i + 1 and its row-sum add at i + 2, and pair q its
  // bf16 pack at 2q + 3 (whole pairs per slot, fma of both at 2q and the
  // rest at 2q + 1 and 2q + 3, measured 1 % slower: the odd slots then carry
  // two exps, the adds and the pack).  With 16 slots (D = 64) score pair p
  // has its fma at slot p, its exp at p + 1 and its pack and adds at p + 3.  A
  // scheduling fence closes every slot, so the exp work stays spread under
  // the MFMAs (each 32x32x16 MFMA leaves room for about two exp and two
  // other VALU instructions of the same SIMD).  The row sum adds the fp32 P
  // values: v_dot2c_f32_bf16 over the packed pair (one instruction instead
  // of two) waits for the SIMD's matrix pipeline on gfx950, about one MFMA
  // per instruction while the other wave's MFMAs run, where adds issue
  // beside them (fp8 at 1152 x 4608: 199.0 -> 191.0 us with the adds).
  // The fully unrolled slot program of the fp8 instances is larger than
  // LLVM's default limit for a pragma-requested full unroll; the library is
  // built with a higher one (-pragma-unroll-threshold), without which the
  // loop stays rolled and its per-slot arrays go to scratch memory.
  constexpr int NS = 4 * DB + 2 * QS;
  constexpr int PREF = 3;
  // fp8 staging inside the slot program: one unit (a K row chunk, a V half,
  // a load) every kStageStride slots from kStageSlot0 on
  constexpr int kStageSlot0 = 0, kStageStride = 1;
  const uint16_t* vf0 = &vbuf[0][vrow(li) + hg * 8];
  const uint16_t* kf0 = &kbuf[0][li * KS + hg * 8];
  auto tile = [&](int vb, int kbf, const f32x16_t (&scur)[2], f32x16_t (&snext)[2], const uint32_t (&pprev)[16],
                  uint32_t (&pcur)[16], float& ps0, float& ps1, float c, float neg_m, auto&& slot_work) {
    const f32x16_t zero = f32x16_t{};
    const uint16_t* vf = vf0 + vb * VBUF;
    const uint16_t* kf = kf0 + kbf * KBUF;
    auto frag = [&](int t) -> bf16x8_t {
      if (t < 4 * DB) return *reinterpret_cast<const bf16x8_t*>(vf + vrow((t % DB) * 32) + (t / DB) * 16);
      const int u = t - 4 * DB;
      return *reinterpret_cast<const bf16x8_t*>(kf + (u & 1) * 32 * KS + (u >> 1) * 16);
    };
    bf16x8_t ring[PREF + 1];
#pragma unroll
    for (int t = 0; t < PREF; ++t) ring[t] = frag(t);
    float e0[16], e1[16];
    ps0 = 0.0f;
    ps1 = 0.0f;
#pragma unroll
    for (int t = 0; t < NS + 2; ++t) {
      if (t < NS) {
        if (t + PREF < NS) ring[(t + PREF) % (PREF + 1)] = frag(t + PREF);
        const bf16x8_t a = ring[t % (PREF + 1)];
        if (t < 4 * DB) {
          const int k4 = t / DB, d = t % DB;
          const bf16x8_t pf = __builtin_bit_cast(
              bf16x8_t, make_uint4(pprev[4 * k4], pprev[4 * k4 + 1], pprev[4 * k4 + 2], pprev[4 * k4 + 3]));
          oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pf, oacc[d], 0, 0, 0);
        } else {
          const int u = t - 4 * DB, kb = u & 1, kk = u >> 1;  // the two key blocks' chains alternate
          snext[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qf[kk], kk == 0 ? zero : snext[kb], 0, 0, 0);
        }
      }
      slot_work(t);
      if constexpr (NS == 32) {
        // one score per slot: its fma at slot i, its exp at i + 1, its
        // row-sum add at i + 2, and the bf16 pack of pair q at 2q + 3, so
        // every slot carries the same vector work
#pragma unroll
        for (int i = 0; i < 32; ++i) {
          const int q = i >> 1, kb = q >> 3, r = (q & 7) * 2 + (i & 1);
          float* e = (i & 1) ? e1 : e0;
          if (t == i) e[q] = __builtin_fmaf(scur[kb][r], c, neg_m);
          if (t == i + 1) e[q] = __builtin_amdgcn_exp2f(e[q]);
          if (t == i + 2) {
            float& ps = (i & 1) ? ps1 : ps0;
            ps = ps + e[q];
          }
        }
#pragma unroll
        for (int q = 0; q < 16; ++q)
          if (t == 2 * q + 3) {
            pcur[q] = pack_bf16x2(e0[q], e1[q]);
            asm volatile("" : "+v"(pcur[q]));
          }
      } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int kb = q >> 3, r = (q & 7) * 2;
          if ((2 * q * NS) / 32 == t) {
            e0[q] = __builtin_fmaf(scur[kb][r], c, neg_m);
            e1[q] = __builtin_fmaf(scur[kb][r + 1], c, neg_m);
          }
          if ((2 * q * NS) / 32 + 1 == t) {
            e0[q] = __builtin_amdgcn_exp2f(e0[q]);
            e1[q] = __builtin_amdgcn_exp2f(e1[q]);
          }
          if ((2 * q * NS) / 32 + 3 == t || (q == 15 && t == NS + 1 && (2 * q * NS) / 32 + 3 > NS + 1)) {
            pcur[q] = pack_bf16x2(e0[q], e1[q]);
            float& ps = (q & 1) ? ps1 : ps0;
            ps = ps + e0[q];
            ps = ps + e1[q];
            // with no use left in this slot the compiler would sink the pack
            // to the next tile's PV and issue all sixteen back to back after
            // the slot program; pin it here, under this slot's MFMA
            asm volatile("" : "+v"(pcur[q]));
          }
        }
      }
      // the slot's order at D = 128: MFMA, fragment read, exp, other vector work.
      // Medians of four alternating runs, without and with it: fp8 1152 x 6912
      // 237.7 and 234.4 us, 1728 x 10368 523.6 and 514.7, in 330-token frames
      // 990 x 5940 234.5 and 229.8 (another box: 240.3 and 238.5, 524.6 and 521.4,
      // 236.7 and 233.0); spilled VGPRs of the fp8 kernels: pair 1 and 0,
      // 4-wave 2 and 0, framed 12 and 6.  At D = 64 the compiler's order is the
      // faster one (fp8 1152 x 6912 167.5 against 169.0 us, bf16 300 x 4500 48.4
      // against 48.9).
      if constexpr (D == 128) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  if (ntiles > 0) {
    f32x16_t sa[2], sb[2];
    uint32_t pa[16], pb[16];  // P(j) of even / odd j
    // ---- prologue: S(0) sets m from its own maximum; P(0); S(1) ----
    int nv0;
    if constexpr (FP8) {
      // K(0), V(0), K(1) decoded into LDS; K(2) and V(1) left in registers
      nv0 = cit.nvalid();
      load_k8();
      load_v8();
      load_q();
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      store_k8(0);
      store_v8(0);
      if (ntiles > 1) {
        load_k8();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        store_k8(1);
        load_v8();
      }
      if (ntiles > 2) load_k8();
      publish();
    } else {
      issue_k(0);
      if (ntiles > 1) issue_k(1);
      nv0 = vit.nvalid();  // valid keys of tile 0 (the V stream is at tile j before V(j) is issued)
      issue_v(0);
      load_q();  // its latency overlaps the first tiles' loads
      publish();
    }
    qk_tile(0, sa);
    if (nv0 < BN) mask_tail(sa, nv0);
    {
      const TileScale ts = tile_scale();
      m_run = tile_max(sa, ts.c);
      l_run = exp_all(sa, pa, ts.c, ts.off - m_run) * ts.inv;
      if constexpr (FP8) cit.next(p.k_ptr, 0, 0, p);
    }
    if (ntiles > 1) qk_tile(1, sb);
    if (ntiles > 2) {
      __syncthreads();  // every wave is done with K(0)
      if constexpr (FP8) {
        store_k8(0);                   // K(2)
        if (ntiles > 3) load_k8();     // K(3)
      } else {
        issue_k(0);                    // K(2)
      }
    }
    // ---- iteration j (1 <= j < ntiles): the slot program computes
    //      O += V(j-1)^T P(j-1), S(j+1) = K(j+1) Q^T and P(j) = 2^(S(j)c - m).
    //      On the last tile S(j+1) is computed from stale LDS and dropped. ----
    auto step = [&](int j, f32x16_t (&scur)[2], f32x16_t (&snext)[2], const uint32_t (&pprev)[16],
                    uint32_t (&pcur)[16]) {
      int nv;
      if constexpr (FP8) {
        // registers hold K(j+2) and V(j); LDS holds K(j+1) and V(j-1)
        publish();  // the buffers of K(j) and V(j-2) are free
        nv = cit.nvalid();
      } else {
        publish();  // K(j+1) and V(j-1) have landed; the buffers of K(j) and V(j-2) are free
        if (j + 2 < ntiles) issue_k(j & 1);  // K(j+2)
        nv = vit.nvalid();                   // valid keys of tile j
        issue_v(j & 1);                      // V(j)
      }
      if (nv < BN) mask_tail(scur, nv);
      const TileScale ts = tile_scale();
      float ps0, ps1;
      // fp8: the decode of K(j+2) and V(j) into the free buffers and the
      // loads of K(j+3) and V(j+1) into the freed registers ride in the slot
      // program, under the matrix work of tile j
      tile((j - 1) & 1, (j + 1) & 1, scur, snext, pprev, pcur, ps0, ps1, ts.c, ts.off - m_run, [&](int t) {
        if constexpr (FP8) {
#pragma unroll
          for (int i = 0; i < FKL; ++i)
            if (t == kStageSlot0 + kStageStride * i && j + 2 < ntiles) store_k8_row(j & 1, i);  // K(j+2)
          if (t == kStageSlot0 + kStageStride * FKL && j + 3 < ntiles) load_k8();               // K(j+3)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh)
            if (t == kStageSlot0 + kStageStride * (FKL + 1 + hh)) store_v8_half(j & 1, hh);     // V(j)
          if (t == kStageSlot0 + kStageStride * (FKL + 3) && j + 1 < ntiles) load_v8();         // V(j+1)
        }
      });
      float ps = (ps0 + ps1) * ts.inv;
      if (__builtin_amdgcn_ballot_w64(ps > kOver)) {
        // raise m to the tile maximum, rescale O and l, redo P(j) from S(j)
        const float m_new = fmaxf(m_run, tile_max(scur, ts.c));
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int d = 0; d < DB; ++d) oacc[d] *= alpha;
        ps = exp_all(scur, pcur, ts.c, ts.off - m_run) * ts.inv;
      }
      l_run += ps;
      if constexpr (FP8) cit.next(p.k_ptr, 0, 0, p);
    };
    int j = 1;
    for (; j + 1 < ntiles; j += 2) {
      step(j, sb, sa, pa, pb);
      step(j + 1, sa, sb, pb, pa);
    }
    if (j < ntiles) step(j, sb, sa, pa, pb);
    // ---- epilogue: O += V(n-1)^T P(n-1) ----
    publish();
    if ((ntiles - 1) & 1)
      pv_tile(1, pb);
    else
      pv_tile(0, pa);
  }

  // output staging: waves 0-3 in the K buffers, the pair kernel's group 1 in the V buffers
  static_assert(4 * 32 * (D + 8) <= 2 * KBUF && 4 * 32 * (D + 8) <= 2 * VBUF, "output staging region");
  const int owave = PAIR ? wave : (int)(threadIdx.x >> 6);
  uint16_t* stage = (PAIR && grp == 1 ? &vbuf[0][0] : &kbuf[0][0]) + owave * 32 * (D + 8);
  finish_tile<D, stores_f32_partials(D, PAIR, false)>(p, wi, b, h, qt, owave * 32 + (int)(threadIdx.x & 31), oacc, m_run, pair_sum(l_run), stage);
}

// KV operands of a kernel instance: bf16 with key-major V (kKeyMajorV32: on
// 32x32x16 MFMAs), bf16 with token-major V, or fp8 (frames of whole 64-key tiles)
enum KvKind { kKeyMajorV, kKeyMajorV32, kTokenMajorV, kFp8 };

template <int D, KvKind KV>
__global__ void __launch_bounds__(256, 2) flash_fwd_pipe_kernel(const FlashParams p) {
  if constexpr (KV == kFp8 || KV == kKeyMajorV32)
    flash_mfma32_body<D, KV == kFp8, false>(p);
  else
    flash_bf16_body<D, false, KV == kTokenMajorV>(p);
}

// an even number of q-tiles per head: pair workgroups
template <int D, KvKind KV>
__global__ void __launch_bounds__(512, 1) flash_fwd_pair_kernel(const FlashParams p) {
  if constexpr (KV == kFp8)
    flash_mfma32_body<D, true, false, true>(p);
  else
    flash_bf16_body<D, true, KV == kTokenMajorV>(p);
}

// fp8 frames that are not a whole number of 64-key tiles
template <int D>
__global__ void __launch_bounds__(256, 2) flash_fwd_pipe_framed_kernel(const FlashParams p) {
  flash_mfma32_body<D, true, true>(p);
}

template <int D>
int launch_combine(const FlashParams& p, hipStream_t st) {
  if (p.split <= 1) return LTX_OK;
  const int64_t tail = (int64_t)p.B * p.H * p.n_qtiles - (p.pair ? 2 * (int64_t)p.n_full : p.n_full);
  const int64_t wg_per_tile = combine_wg_per_tile<D>();
  const dim3 grid((unsigned)(tail * wg_per_tile));
  if (p.part_f32)
    hipLaunchKernelGGL((flash_combine_kernel<D, true>), grid, dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((flash_combine_kernel<D, false>), grid, dim3(256), 0, st, p);
  LTX_LAUNCH_CHECK("ltx_flash_attn_fwd (combine)");
  return LTX_OK;
}

// Grid: whole q-tiles (pair kernel: units of two) first, then the key-range
// pieces of the tail ones.
inline int64_t grid_blocks(const FlashParams& p) {
  const int64_t nq = (int64_t)p.B * p.H * p.n_qtiles / (p.pair ? 2 : 1);
  return p.n_full + (nq - p.n_full) * p.split;
}

template <int D, KvKind KV, bool FRAMED = false>
int launch_flash_pipe(const FlashParams& p, hipStream_t st) {
  static_assert(KV == kFp8 || !FRAMED, "frame tiling is an fp8 feature");
  const int64_t nblocks = grid_blocks(p);
  LTX_REQUIRE(nblocks <= 0x7FFFFFFF, "ltx_flash_attn_fwd: grid too large");
  if constexpr (FRAMED)
    hipLaunchKernelGGL((flash_fwd_pipe_framed_kernel<D>), dim3((unsigned)nblocks), dim3(256), 0, st, p);
  else if (KV != kKeyMajorV32 && p.pair)
    hipLaunchKernelGGL((flash_fwd_pair_kernel<D, KV == kKeyMajorV32 ? kKeyMajorV : KV>), dim3((unsigned)nblocks), dim3(512), 0, st, p);
  else
    hipLaunchKernelGGL((flash_fwd_pipe_kernel<D, KV>), dim3((unsigned)nblocks), dim3(256), 0, st, p);
  LTX_LAUNCH_CHECK("ltx_flash_attn_fwd");
  return launch_combine<D>(p, st);
}

template <int D>
int launch_flash_masked(const FlashParams& p, hipStream_t st) {
  const int64_t nblocks = grid_blocks(p);
  LTX_REQUIRE(nblocks <= 0x7FFFFFFF, "ltx_flash_attn_fwd: grid too large");
  hipLaunchKernelGGL((flash_fwd_masked_kernel<D>), dim3((unsigned)nblocks), dim3(256), 0, st, p);
  LTX_LAUNCH_CHECK("ltx_flash_attn_fwd");
  return launch_combine<D>(p, st);
}

}  // namespace ltx

using namespace ltx;

// Resident workgroups the device holds for this kernel (CUs x occupancy),
// computed once per device under a once-flag (calls from several host
// threads may race to fill it); one table per kernel (each instantiation of
// the template has its own).
constexpr int kMaxDevices = 64;
struct Slots {
  int slots;  // resident workgroups (0: unknown, no split is planned)
  int cus;
};
template <auto Kernel>
Slots resident_slots(int threads = 256) {
  static std::once_flag once[kMaxDevices];
  static Slots slots[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return Slots{0, 1};
  std::call_once(once[dev], [&]() {
    int cus = 0, occ = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, Kernel, threads, 0) != hipSuccess) {
      slots[dev] = Slots{0, 1};
      return;
    }
    occ = occ > 0 ? occ : 1;
    slots[dev] = Slots{cus * occ, cus};
  });
  return slots[dev];
}

// The kernel family a call takes: the masked staged kernel for a key mask,
// else the pipelined one of its KV kind (the pair instance when the q-tiles
// per head are even; fp8 framed shares the pipelined kernel's occupancy).
enum FlashPath { kPathKeyMajor, kPathTokenMajor, kPathFp8, kPathMasked };

template <int D>
Slots slots_for(FlashPath path, bool pair) {
  switch (path) {
    case kPathKeyMajor:
      return pair ? resident_slots<flash_fwd_pair_kernel<D, kKeyMajorV>>(512)
                  : resident_slots<flash_fwd_pipe_kernel<D, kKeyMajorV>>();
    case kPathTokenMajor:
      return pair ? resident_slots<flash_fwd_pair_kernel<D, kTokenMajorV>>(512)
                  : resident_slots<flash_fwd_pipe_kernel<D, kTokenMajorV>>();
    case kPathFp8:
      return pair ? resident_slots<flash_fwd_pair_kernel<D, kFp8>>(512)
                  : resident_slots<flash_fwd_pipe_kernel<D, kFp8>>();
    default:
      return resident_slots<flash_fwd_masked_kernel<D>>();
  }
}
inline Slots flash_slots(int64_t D, FlashPath path, bool pair) {
  return D == 128 ? slots_for<128>(path, pair) : slots_for<64>(path, pair);
}

struct Split {
  int64_t n_full;  // work units that run whole
  int n;           // key ranges of each of the others
  bool f32;        // the ranges' partial O in float32
  // partial rows of `units` work units of `per_unit` q-tiles, and their bytes:
  // (max, sum) in float32 for every row, then the O rows
  int64_t rows(int64_t units, int per_unit) const { return n > 1 ? (units - n_full) * per_unit * n * kBM : 0; }
  int64_t bytes(int64_t units, int per_unit, int64_t D) const {
    return rows(units, per_unit) * (2 * 4 + D * (f32 ? 4 : 2));
  }
};

// Which work units (q-tiles, or the pair kernel's units of two) are cut into
// key ranges, and into how many.  Whole rounds of resident workgroups run whole;
// the rest, the tail, is cut so that its workgroups spread over the CUs.  Pieces
// keep >= 4 key tiles behind a whole round, >= 2 in a grid that is a single
// partial round (the 75-query audio and V2A calls: V2A 75 x 1152 16.0 -> 12.5
// us, audio self-attention 75 x 675 14.2 -> 12.6 us).
//
// Base: one piece per CU.  Of the workgroups one CU holds, the oldest one's
// waves win the issue arbitration: with two 4-wave workgroups per CU the older
// finishes its q-tile about a quarter before the younger, so one slot per CU
// frees early.  Pieces that fill just those slots run beside the younger
// workgroups' last stretch; pieces for every slot leave their second half to
// start only when the younger workgroups end (1152 x 4608 bf16: 193.7 against
// 184.8 us for the step with 8 against 4 pieces per tail q-tile; fp8 187.6
// against 180.4 us).  The masked kernel's pieces fill every slot.  The pair
// kernel keeps to the base: at 6, 12 and 14 q-tiles per head its partly filled
// rounds measured no slower than any split.
//
// What may be split further is bounded by exactness.  A range's O is rounded to
// bf16 before the merge, which makes the error against float64 1.22 times the
// whole call's where all rows are split; over more ranges it averages out a
// little.  So units that the base leaves whole (a tail of more than half the
// CUs) keep their float32 sums: they are split only with float32 partials
// (0.96 to 1.003 times the whole call's error), whose traffic (25 MB written and
// read again for 384 pieces at D = 128) costs 10 to 15 us, and so only over
// enough keys.  Measured in us, whole against
// split, by tail and ranges (B * H = 16 to 64 heads; KT key tiles, for fp8 KT
// tiles in 330-token frames):
//   up to 1/3 of the slots, 3 ranges: bf16 D = 128 tail 160 at KT 41: 38.6 / 40.2,
//     54: 48.2 / 45.4, 162: 133 / 103; D = 64 at 41: 30.1 / 28.3, 108: 70.3 / 48.9;
//     fp8 at 24: 41.4 / 38.6, 84: 125 / 78
//   up to 1/2, 2 ranges, or 4 where those fill at most 1.5 rounds: tail 192 D = 128
//     at 72: 64.2 / 68.5, 108: 94.0 / 98.1, 162: 194 / 137; D = 64 at 72: 48.9 / 43.4,
//     108: 70.9 / 58.1; fp8 at 24: 41.5 / 44.3, 36: 59.1 / 55.7, 84: 127 / 97
//   up to 2/3, 3 ranges: tail 320 D = 128 at 54: 81.8 / 83.3, 72: 107 / 103, 162: 235 / 211;
//     fp8 at 36: 79.5 / 81.4, 48: 102 / 97; token-major at 54: 89.2 / 87.1
//   up to 3/4, 2 ranges: tail 352 D = 128 at 72: 109 / 110, 108: 161 / 155; fp8 at 48:
//     102 / 105, 84: 171 / 164
//   above: no split gains (tail 416 and 448: 1.03 to 1.3 times as long up to 6912 keys)
// More ranges in bf16 than the base cost no exactness: grids of one partial
// round take one piece per slot where the base gives 2 or 3 ranges (fp8: 4 too)
// and the keys are long.  Base / one per slot: tail 96 (2 / 5 ranges) D = 128 at KT
// 41: 28.3 / 27.8, 54: 33.0 / 30.7; D = 64 at 21: 16.4 / 16.3, 31: 19.5 / 17.7; fp8 at 24: 29.9 /
// 26.5, 48: 46.5 / 35.9; tail 112 (2 / 4) D = 128 at 41: 29.5 / 30.2, 54: 33.9 / 33.7; tail 72
// (3 / 7) D = 128 at 41: 23.7 / 24.6, 63: 29.7 / 29.2; D = 64 at 31: 16.7 / 17.3, 41: 18.8 /
// 18.1; fp8 at 24: 24.8 / 25.0, 36: 30.4 / 28.4.
//
// Token-major calls came from a staged kernel whose pieces filled every slot
// (three workgroups per CU at D = 64, where up to 768 q-tiles were one round).  In
// a partial round they keep at least as many bf16 ranges (V2A 75 x 1152: error
// 1.020 times with 4 instead of 8), or run whole over few keys (tail 160 at D = 128,
// whole / 3 ranges, KT 27: 34.0 / 29.4; tail 192, whole / 2, 41: 48.6 / 46.2), or,
// at D = 64, take float32 partials where fewer ranges are faster:
//   tails up to 64: 8 bf16 ranges (tail 64 at KT 18: 14.4, 4 in float32 15.2)
//   more: one piece per CU in float32, per slot over longer keys (tail 80, 3 / 5
//     ranges, KT 41: 21.9 / 25.5, 162: 49.2 / 46.8; tail 96, 2 / 5, 41: 25.9 / 24.5,
//     72: 35.2 / 29.3; tail 160, whole / 3, 27: 24.3 / 24.8, 41: 34.4 / 29.8), whole over
//     few keys (tail 80, whole / 3, 11: 13.5 / 14.9, 18: 18.0 / 16.0; 128 pair units,
//     whole / 2, 15: 22.3 / 27.5)
//   a third to a half of the slots: the bf16 ranges of three per CU (tail 192, 4 bf16
//     / 2 float32, KT 41: 32.5 / 34.8, 162: 83.8 / 97.1)
// Behind whole rounds four bf16 ranges are as exact as eight (1.0005) at D = 128; two
// or three are not, nor any at D = 64, whose rows ran whole there.  (The pair units'
// ranges at D = 128 are the ones that the staged kernel had.)
inline Split plan_split(int64_t units, int ntiles, FlashPath path, bool pair, int64_t D) {
  const Slots s = flash_slots(D, path, pair);
  if (s.slots <= 0 || units % s.slots == 0) return {units, 1, false};
  const int64_t S = s.slots, full = units / S * S, tail = units - full;
  const bool one_round = full == 0, token = path == kPathTokenMajor, fp8 = path == kPathFp8, d64 = D == 64;
  const bool two_per_cu = !pair && path != kPathMasked && S == 2 * s.cus;
  auto below = [](int64_t n, int64_t limit) { return n < limit ? n : limit; };

  int64_t n = (path == kPathMasked ? S : s.cus) / tail;
  bool f32 = false;
  if (token && one_round) {
    const int64_t least = d64 ? (S + S / 2) / tail : S / tail;
    if (!d64 || (two_per_cu && (4 * tail <= s.cus || (3 * tail > S && 2 * tail <= S))))
      n = least;
    else if (two_per_cu && ntiles >= (n >= 3 ? 128 : n == 2 ? 48 : 36))
      n = S / tail;
    f32 = n < below(least, kMaxSplit);
    if (two_per_cu && 2 * tail > s.cus && ntiles < (d64 || 3 * tail > S ? 36 : 24)) n = 1;
    if (f32 && ntiles < (2 * tail < s.cus || two_per_cu ? 16 : 27)) n = 1;
  } else if (token) {
    f32 = d64 || (two_per_cu && n < 4);
  } else if (two_per_cu && one_round && n >= 2 && n <= (fp8 ? 4 : 3)) {
    if (ntiles >= (n == 2 ? (fp8 ? 24 : d64 ? 32 : 54) : (fp8 ? 36 : d64 ? 40 : 72))) n = S / tail;
  }
  if (two_per_cu && n < 2) {
    f32 = true;
    if (3 * tail <= S)
      n = ntiles >= (fp8 ? 24 : d64 ? 40 : 54) ? 3 : 1;
    else if (2 * tail <= S)
      n = ntiles < (fp8 ? 36 : d64 ? 72 : 128) ? 1 : 8 * tail <= 3 * S && ntiles >= 54 ? 4 : 2;
    else if (3 * tail <= 2 * S)
      n = ntiles >= (fp8 ? 48 : token ? 54 : 72) ? 3 : 1;
    else if (4 * tail <= 3 * S)
      n = ntiles >= (fp8 ? 66 : 100) ? 2 : 1;
  }
  n = below(below(n, kMaxSplit), ntiles / (one_round ? 2 : 4));
  return n >= 2 ? Split{full, (int)n, f32} : Split{units, 1, false};
}

inline int64_t round256(int64_t x) { return (x + 255) / 256 * 256; }

// Key-major bf16 calls that keep the 32x32x16 kernel: the 4-wave kernel with
// up to 11/8 workgroups per CU, or fewer than 16 key tiles.  The CUs
// then hold one wave per SIMD for much of the call, the part is not power
// bound, and a wave issues half as many MFMAs: 32.7 against 35.5 us for 3
// q-tiles per head over 2048 keys (B = 2, 32 heads x 128: 192 workgroups), 70.5
// against 73.8 us for 5 over 4608 keys at 32 x 64 (320), 30.1
// against 31.5 us for 11 over 1728 keys at B = 1 (352), and 26.0 against 27.4
// us for 9 over 832 keys.  With 448 workgroups the 16x16x32 kernel leads
// again (126.9 against 130.2 us, 7 over 4608 keys).
inline bool small_grid(const FlashParams& p, Slots s) {
  return !p.pair && (p.tile_start[p.n_seg] < 16 || 8 * grid_blocks(p) <= 11 * (int64_t)s.cus);
}

// fp8 K/V in frames of whole 64-key tiles with an odd number (>= 3) of
// q-tiles per head runs as two launches: the first n_qtiles - 1 q-tiles of
// every head as pair workgroups (each thread stages half of a K/V tile that
// two q-tiles share), then the last q-tile of every head on the 4-wave
// kernel, cut into key ranges so that its workgroups fill every slot (they
// start on an empty GPU, so two per CU beat one), merged by the combine
// kernel.  At 1152 queries over 4608 keys (B = 2, 32 heads) that is 256 pair
// units in one round and 64 q-tiles in 8 ranges of 9 key tiles.  SplitPlan
// holds both launches' split plans and their partial buffers' offsets.
struct SplitPlan {
  Split s[2];
  int64_t off[2];
  int64_t total;
};

inline SplitPlan plan_fp8_split_launch(int64_t B, int64_t H, int64_t nqt, int ntiles, int64_t D) {
  SplitPlan sp{};
  // launch 0: pair units over the first nqt - 1 q-tiles of every head
  const int64_t nu0 = B * H * (nqt - 1) / 2;
  sp.s[0] = plan_split(nu0, ntiles, kPathFp8, true, D);
  // launch 1: the last q-tile of every head, one piece per slot
  const int64_t nu1 = B * H;
  const Slots s1 = flash_slots(D, kPathFp8, false);
  sp.s[1] = {nu1, 1, false};
  if (s1.slots > 0 && nu1 < s1.slots) {
    int k = (int)(s1.slots / nu1);
    k = k > kMaxSplit ? kMaxSplit : k;
    k = k > ntiles / 2 ? ntiles / 2 : k;   // pieces of >= 2 key tiles
    if (k >= 2) sp.s[1] = {0, k, false};
  }
  sp.off[0] = 0;
  sp.off[1] = round256(sp.s[0].bytes(nu0, 2, D));
  sp.total = sp.off[1] + sp.s[1].bytes(nu1, 1, D);
  return sp;
}

extern "C" int ltx_flash_attn_workspace_size(int64_t B, int64_t Lq, int64_t H, int64_t D,
                                             int64_t* bytes) {
  clear_error();
  LTX_REQUIRE(bytes != nullptr && B >= 1 && H >= 1 && Lq >= 0 && (D == 64 || D == 128),
              "ltx_flash_attn_workspace_size: bad arguments");
  // the largest partial buffer any of the kernels for this D may plan (the
  // pair kernel plans over units of two q-tiles)
  const int64_t nqt = (Lq + kBM - 1) / kBM;
  const int64_t nq = B * H * nqt;
  const bool pair = nqt % 2 == 0;
  int64_t need = 0;
  // (fp8 in frames that are not whole tiles takes single q-tiles at an even
  // count too)
  for (int k = 0; k < 5; ++k) {
    const FlashPath path = k == 4 ? kPathFp8 : (FlashPath)k;
    const bool kp = pair && k != 4 && path != kPathMasked;
    const int64_t nu = kp ? nq / 2 : nq;
    // no call of this shape plans more than one with an unbounded key count
    const int64_t b = plan_split(nu, 1 << 30, path, kp, D).bytes(nu, kp ? 2 : 1, D);
    need = b > need ? b : need;
  }
  // the two-launch fp8 plan for an odd q-tile count
  if (nqt >= 3 && nqt % 2 == 1) {
    const int64_t b = plan_fp8_split_launch(B, H, nqt, 1 << 30, D).total;
    need = b > need ? b : need;
  }
  *bytes = need;
  return LTX_OK;
}

// The body of the attention entry points.  A planned split whose partials do
// not fit the workspace runs whole.  `seg_bs`: each segment's own batch stride (in
// elements, instead of k_bs), for token-major bf16 K/V.
static int flash_attn_fwd_impl(const void* q, int64_t B, int64_t Lq, int64_t H, int64_t D,
                               int64_t q_bs, int64_t q_ls, int64_t q_hs, int64_t n_segments,
                               const void* const* k_ptrs, const void* const* v_ptrs,
                               const int64_t* seg_lens, int64_t k_bs, int64_t k_ls, int64_t k_hs,
                               int64_t v_bs, int64_t v_ls, int64_t v_hs, int64_t v_ds, int kv_dtype,
                               const float* const* k_scales, const float* const* v_scales,
                               int64_t sc_bs, int64_t sc_hs, int64_t frame_tokens,
                               const float* key_mask, int64_t mask_bs, const int64_t* key_lens, void* out,
                               int64_t o_bs, int64_t o_ls, int64_t o_hs, float* lse, float scale,
                               void* workspace, int64_t workspace_bytes, void* stream,
                               const int64_t* seg_bs = nullptr) {
  LTX_REQUIRE(q && out, "ltx_flash_attn_fwd: null q/out");
  LTX_REQUIRE(D == 64 || D == 128, "ltx_flash_attn_fwd: head dim %lld unsupported (64 or 128)",
              (long long)D);
  LTX_REQUIRE(B >= 1 && H >= 1 && Lq >= 0 && Lq <= 0x7FFFFFFF, "ltx_flash_attn_fwd: bad B/H/Lq");
  LTX_REQUIRE(n_segments >= 0 && n_segments <= LTX_MAX_SEGMENTS,
              "ltx_flash_attn_fwd: n_segments must be in [0, %d]", LTX_MAX_SEGMENTS);
  LTX_REQUIRE(kv_dtype == LTX_BF16 || kv_dtype == LTX_F8E4M3, "ltx_flash_attn_fwd: kv_dtype must be BF16 or F8E4M3");
  LTX_REQUIRE(n_segments == 0 || (k_ptrs && v_ptrs && seg_lens), "ltx_flash_attn_fwd: null segment arrays");
  const bool fp8 = kv_dtype == LTX_F8E4M3;
  const bool vkey = v_ds != 1;  // key-major V
  LTX_REQUIRE(!vkey || v_ls == 1, "ltx_flash_attn_fwd: V must be token-major (v_ds == 1) or key-major (v_ls == 1)");
  LTX_REQUIRE(!vkey || (!fp8 && key_mask == nullptr),
              "ltx_flash_attn_fwd: key-major V is bf16 without a key mask");
  const int64_t esz = fp8 ? 1 : 2;
  auto al = [](const void* ptr, uintptr_t a) { return ((uintptr_t)ptr % a) == 0; };
  LTX_REQUIRE(al(q, 16) && (q_bs * 2) % 16 == 0 && (q_ls * 2) % 16 == 0 && (q_hs * 2) % 16 == 0,
              "ltx_flash_attn_fwd: q rows must be 16-byte aligned");
  LTX_REQUIRE(al(out, 8) && (o_bs * 2) % 8 == 0 && (o_ls * 2) % 8 == 0 && (o_hs * 2) % 8 == 0,
              "ltx_flash_attn_fwd: out rows must be 8-byte aligned");
  LTX_REQUIRE((k_bs * esz) % 16 == 0 && (k_ls * esz) % 16 == 0 && (k_hs * esz) % 16 == 0,
              "ltx_flash_attn_fwd: K strides must keep 16-byte rows");
  if (vkey)
    LTX_REQUIRE((v_bs * 2) % 16 == 0 && (v_hs * 2) % 16 == 0 && (v_ds * 2) % 16 == 0 &&
                    v_ds * D * 2 < ((int64_t)1 << 31),
                "ltx_flash_attn_fwd: key-major V strides must keep 16-byte rows");
  else
    LTX_REQUIRE(v_bs == k_bs && v_ls == k_ls && v_hs == k_hs,
                "ltx_flash_attn_fwd: token-major V must share K's strides");

  FlashParams p{};
  p.q = (const uint16_t*)q;
  p.o = (uint16_t*)out;
  p.lse = lse;
  p.mask = key_mask;
  p.q_bs = q_bs; p.q_ls = q_ls; p.q_hs = q_hs;
  p.o_bs = o_bs; p.o_ls = o_ls; p.o_hs = o_hs;
  p.o_al16 = ((uintptr_t)out % 16 == 0 && o_bs % 8 == 0 && o_ls % 8 == 0 && o_hs % 8 == 0) ? 1 : 0;
  p.kv_ls = k_ls; p.kv_hs = k_hs;
  p.v_bs = v_bs; p.v_hs = v_hs; p.v_ds = v_ds;
  p.sc_bs = sc_bs; p.sc_hs = sc_hs;
  p.mask_bs = mask_bs;
  p.B = (int)B; p.H = (int)H; p.Lq = (int)Lq;
  p.frame = (int)(frame_tokens > 0 ? frame_tokens : 1);
  p.scale = scale > 0.0f ? scale : 1.0f / sqrtf((float)D);
  p.scale_log2 = p.scale * kLog2e;
  // drop empty segments
  int n = 0;
  p.seg_start[0] = 0;
  p.tile_start[0] = 0;
  for (int64_t i = 0; i < n_segments; ++i) {
    LTX_REQUIRE(seg_lens[i] >= 0, "ltx_flash_attn_fwd: negative segment length");
    if (seg_lens[i] == 0) continue;
    LTX_REQUIRE(k_ptrs[i] && v_ptrs[i], "ltx_flash_attn_fwd: null segment %lld", (long long)i);
    LTX_REQUIRE(al(k_ptrs[i], 16) && al(v_ptrs[i], 16), "ltx_flash_attn_fwd: segment %lld not 16-byte aligned",
                (long long)i);
    if (fp8) {
      LTX_REQUIRE(k_scales && v_scales && k_scales[i] && v_scales[i],
                  "ltx_flash_attn_fwd: fp8 segment %lld needs k/v scales", (long long)i);
      LTX_REQUIRE(frame_tokens > 0 && frame_tokens <= 0x7FFFFFFF,
                  "ltx_flash_attn_fwd: fp8 needs frame_tokens > 0 (got %lld)", (long long)frame_tokens);
      p.k_sc[n] = k_scales[i];
      p.v_sc[n] = v_scales[i];
    }
    const int64_t bs = seg_bs != nullptr ? seg_bs[i] : k_bs;
    LTX_REQUIRE((bs * esz) % 16 == 0, "ltx_flash_attn_fwd: segment %lld's batch stride must keep 16-byte rows",
                (long long)i);
    p.seg_bs[n] = bs * esz;
    p.k_ptr[n] = k_ptrs[i];
    p.v_ptr[n] = v_ptrs[i];
    p.seg_start[n + 1] = p.seg_start[n] + seg_lens[i];
    // fp8: tiles never cross a frame (ceil(F / 64) per frame, the segment's
    // last frame possibly partial); bf16: ceil(len / 64)
    const int64_t seg_tiles =
        fp8 ? (seg_lens[i] / frame_tokens) * ((frame_tokens + kBN - 1) / kBN) +
                  (seg_lens[i] % frame_tokens + kBN - 1) / kBN
            : (seg_lens[i] + kBN - 1) / kBN;
    const int64_t tiles = p.tile_start[n] + seg_tiles;
    LTX_REQUIRE(tiles <= 0x7FFFFFFF, "ltx_flash_attn_fwd: too many keys");
    p.tile_start[n + 1] = (int)tiles;
    ++n;
  }
  p.n_seg = n;
  p.Lk = p.seg_start[n];
  if (key_mask) LTX_REQUIRE(!fp8, "ltx_flash_attn_fwd: key mask with fp8 KV is not built");
  if (key_lens) {
    LTX_REQUIRE(vkey && !fp8 && key_mask == nullptr,
                "ltx_flash_attn_fwd: key_lens needs bf16 key-major V and no key mask");
    LTX_REQUIRE(B <= LTX_MAX_KEYLEN_BATCH, "ltx_flash_attn_fwd: key_lens supports at most %d batch rows",
                LTX_MAX_KEYLEN_BATCH);
    for (int64_t b = 0; b < B; ++b) {
      LTX_REQUIRE(key_lens[b] >= 0 && key_lens[b] <= p.Lk,
                  "ltx_flash_attn_fwd: key_lens[%lld] = %lld outside [0, %lld]", (long long)b,
                  (long long)key_lens[b], (long long)p.Lk);
      p.klen[b] = (int)key_lens[b];
    }
    p.n_klen = (int)B;
  }
  LTX_REQUIRE(k_ls * esz * kBN < (int64_t)1 << 31 && k_ls >= D,
              "ltx_flash_attn_fwd: kv token stride %lld out of range", (long long)k_ls);
  p.n_qtiles = (int)((Lq + kBM - 1) / kBM);
  if (Lq == 0) return LTX_OK;
  LTX_REQUIRE(n > 0, "ltx_flash_attn_fwd: no keys (Lk == 0)");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // fp8 K/V, frames of whole tiles, an odd q-tile count >= 3: two launches
  // (plan_fp8_split_launch), each over its own rows of q and out (q and out
  // offset, Lq cut), so only without lse, whose rows are Lq apart.  A plan
  // whose partials do not fit the workspace takes the one-launch path below.
  if (fp8 && frame_tokens % kBN == 0 && p.n_qtiles >= 3 && p.n_qtiles % 2 == 1 && lse == nullptr &&
      workspace != nullptr) {
    const SplitPlan sp = plan_fp8_split_launch(B, H, p.n_qtiles, p.tile_start[n], D);
    if (sp.total <= workspace_bytes) {
      LTX_REQUIRE(al(workspace, 256), "ltx_flash_attn_fwd: workspace must be 256-byte aligned");
      const int64_t lq0 = (int64_t)(p.n_qtiles - 1) * kBM, nq0 = (int64_t)B * H * (p.n_qtiles - 1);
      FlashParams lp[2] = {p, p};
      lp[0].Lq = (int)lq0;
      lp[0].n_qtiles = p.n_qtiles - 1;
      lp[0].pair = 1;
      lp[1].q = p.q + lq0 * q_ls;
      lp[1].o = p.o + lq0 * o_ls;
      lp[1].o_al16 = ((uintptr_t)lp[1].o % 16 == 0 && o_bs % 8 == 0 && o_ls % 8 == 0 && o_hs % 8 == 0) ? 1 : 0;
      lp[1].Lq = (int)(Lq - lq0);
      lp[1].n_qtiles = 1;
      lp[1].pair = 0;
      for (int i = 0; i < 2; ++i) {
        lp[i].n_full = (int)sp.s[i].n_full;
        lp[i].split = sp.s[i].n;
        lp[i].part_f32 = sp.s[i].f32;
        const int64_t rows = sp.s[i].rows(i == 0 ? nq0 / 2 : (int64_t)B * H, i == 0 ? 2 : 1);
        lp[i].part_ml = reinterpret_cast<float*>(static_cast<char*>(workspace) + sp.off[i]);
        lp[i].part_o = lp[i].part_ml + 2 * rows;
        const int rc = D == 128 ? launch_flash_pipe<128, kFp8>(lp[i], st) : launch_flash_pipe<64, kFp8>(lp[i], st);
        if (rc != LTX_OK) return rc;
      }
      return LTX_OK;
    }
  }
  // balanced tail (needs a workspace; without one every q-tile runs whole).
  // Without a key mask (and, for fp8 K/V, in frames of whole 64-key tiles) an
  // even number of q-tiles per head runs the pair kernel, whose grid counts
  // units of two q-tiles (two partial results per split unit).
  const FlashPath path = key_mask != nullptr ? kPathMasked : fp8 ? kPathFp8 : vkey ? kPathKeyMajor : kPathTokenMajor;
  {
    const int64_t nq = (int64_t)B * H * p.n_qtiles;
    LTX_REQUIRE(nq <= 0x7FFFFFFF, "ltx_flash_attn_fwd: grid too large");
    p.pair = path != kPathMasked && (!fp8 || frame_tokens % kBN == 0) && p.n_qtiles % 2 == 0 ? 1 : 0;
    const int64_t nu = p.pair ? nq / 2 : nq;
    const int per_unit = p.pair ? 2 : 1;
    Split sp{nu, 1, false};
    if (workspace != nullptr) {
      sp = plan_split(nu, p.tile_start[n], path, p.pair != 0, D);
      if (sp.bytes(nu, per_unit, D) > workspace_bytes) sp = {nu, 1, false};
      LTX_REQUIRE(!sp.f32 || stores_f32_partials((int)D, p.pair != 0, path == kPathTokenMajor),
                  "ltx_flash_attn_fwd: a launch plan with float32 partials that its kernel does not store");
    }
    p.n_full = (int)sp.n_full;
    p.split = sp.n;
    p.part_f32 = sp.f32;
    if (sp.n > 1) {
      LTX_REQUIRE(al(workspace, 256), "ltx_flash_attn_fwd: workspace must be 256-byte aligned");
      p.part_ml = static_cast<float*>(workspace);
      p.part_o = p.part_ml + 2 * sp.rows(nu, per_unit);
    }
  }
  switch (path) {
    case kPathKeyMajor:
      if (small_grid(p, flash_slots(D, path, p.pair != 0)))
        return D == 128 ? launch_flash_pipe<128, kKeyMajorV32>(p, st) : launch_flash_pipe<64, kKeyMajorV32>(p, st);
      return D == 128 ? launch_flash_pipe<128, kKeyMajorV>(p, st) : launch_flash_pipe<64, kKeyMajorV>(p, st);
    case kPathTokenMajor:
      return D == 128 ? launch_flash_pipe<128, kTokenMajorV>(p, st) : launch_flash_pipe<64, kTokenMajorV>(p, st);
    case kPathFp8:
      // the framed instances share the plain ones' occupancy (same registers
      // and LDS), so the split plan above holds for them too
      if (frame_tokens % kBN != 0)
        return D == 128 ? launch_flash_pipe<128, kFp8, true>(p, st) : launch_flash_pipe<64, kFp8, true>(p, st);
      return D == 128 ? launch_flash_pipe<128, kFp8>(p, st) : launch_flash_pipe<64, kFp8>(p, st);
    default:
      return D == 128 ? launch_flash_masked<128>(p, st) : launch_flash_masked<64>(p, st);
  }
}

extern "C" int ltx_flash_attn_fwd(const void* q, int64_t B, int64_t Lq, int64_t H, int64_t D,
                                  int64_t q_bs, int64_t q_ls, int64_t q_hs, int64_t n_segments,
                                  const void* const* k_ptrs, const void* const* v_ptrs,
                                  const int64_t* seg_lens, int64_t k_bs, int64_t k_ls, int64_t k_hs,
                                  int64_t v_bs, int64_t v_ls, int64_t v_hs, int64_t v_ds, int kv_dtype,
                                  const float* const* k_scales, const float* const* v_scales,
                                  int64_t sc_bs, int64_t sc_hs, int64_t frame_tokens,
                                  const float* key_mask, int64_t mask_bs, const int64_t* key_lens, void* out,
                                  int64_t o_bs, int64_t o_ls, int64_t o_hs, float* lse, float scale,
                                  void* workspace, int64_t workspace_bytes, void* stream) {
  clear_error();
  return flash_attn_fwd_impl(q, B, Lq, H, D, q_bs, q_ls, q_hs, n_segments, k_ptrs, v_ptrs, seg_lens, k_bs,
                             k_ls, k_hs, v_bs, v_ls, v_hs, v_ds, kv_dtype, k_scales, v_scales, sc_bs, sc_hs,
                             frame_tokens, key_mask, mask_bs, key_lens, out, o_bs, o_ls, o_hs, lse, scale,
                             workspace, workspace_bytes, stream);
}

extern "C" int ltx_flash_attn_fwd_plain(const void* q, int64_t B, int64_t Lq, int64_t H, int64_t D, int64_t q_bs,
                                        int64_t q_ls, int64_t q_hs, int64_t n_segments, const void* const* k_ptrs,
                                        const void* const* v_ptrs, const int64_t* seg_lens, const int64_t* seg_bs,
                                        int64_t kv_ls, int64_t kv_hs, void* out, int64_t o_bs, int64_t o_ls,
                                        int64_t o_hs, float* lse, float scale, void* workspace,
                                        int64_t workspace_bytes, void* stream) {
  clear_error();
  LTX_REQUIRE(n_segments == 0 || seg_bs != nullptr, "ltx_flash_attn_fwd_plain: null segment batch strides");
  return flash_attn_fwd_impl(q, B, Lq, H, D, q_bs, q_ls, q_hs, n_segments, k_ptrs, v_ptrs, seg_lens, 0, kv_ls, kv_hs,
                             0, kv_ls, kv_hs, 1, LTX_BF16, nullptr, nullptr, 0, 0, 0, nullptr, 0, nullptr, out, o_bs,
                             o_ls, o_hs, lse, scale, workspace, workspace_bytes, stream, seg_bs);
}

// ---------------------------------------------------------------------------
// No-allocation variant: the split partials live in a fixed device array.
//
// `scratch` holds the partial results of the split tail q-tiles (per piece:
// 128 rows of (max, sum) in float32 and an O row in bf16 or float32): 384
// float32 pieces at D = 128 or 768 at D = 64, and every bf16 plan of one launch
// (at most 512 pieces at D = 128).  A float32 plan that needs more runs whole,
// and the fp8 two-launch plan, which keeps both launches' partials, is taken
// only where they fit (else one launch).  Every piece writes its whole partial
// before the combine kernel reads it, so nothing needs clearing between calls.
// Each device holds its own copy of the array for the life of the process; its
// device address is looked up once per device (hipGetSymbolAddress) and
// only that address is handed to kernels.  Calls that overlap in time on one
// device share the array and race.
// ---------------------------------------------------------------------------
constexpr int64_t kScratchBytes = LTX_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices];

// The current device's address of `scratch` (nullptr and an error message on failure).
static void* scratch_for_current_device() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("ltx_flash_attn_fwd_noalloc: no current HIP device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
      set_error("ltx_flash_attn_fwd_noalloc: hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}

extern "C" int ltx_flash_attn_fwd_noalloc(const void* q, int64_t B, int64_t Lq, int64_t H, int64_t D,
                                          int64_t q_bs, int64_t q_ls, int64_t q_hs, int64_t n_segments,
                                          const void* const* k_ptrs, const void* const* v_ptrs,
                                          const int64_t* seg_lens, int64_t k_bs, int64_t k_ls, int64_t k_hs,
                                          int64_t v_bs, int64_t v_ls, int64_t v_hs, int64_t v_ds,
                                          int kv_dtype, const float* const* k_scales,
                                          const float* const* v_scales, int64_t sc_bs, int64_t sc_hs,
                                          int64_t frame_tokens, const float* key_mask, int64_t mask_bs,
                                          const int64_t* key_lens, void* out, int64_t o_bs, int64_t o_ls,
                                          int64_t o_hs, float* lse, float scale, void* stream) {
  clear_error();
  void* ws = scratch_for_current_device();
  if (ws == nullptr) return LTX_ELAUNCH;
  return flash_attn_fwd_impl(q, B, Lq, H, D, q_bs, q_ls, q_hs, n_segments, k_ptrs, v_ptrs, seg_lens, k_bs,
                             k_ls, k_hs, v_bs, v_ls, v_hs, v_ds, kv_dtype, k_scales, v_scales, sc_bs, sc_hs,
                             frame_tokens, key_mask, mask_bs, key_lens, out, o_bs, o_ls, o_hs, lse, scale, ws,
                             kScratchBytes, stream);
}
