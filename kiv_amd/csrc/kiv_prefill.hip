// MFMA attention for queries of many positions: prefill chunks and
// multi-position queries over [retrieved ; hot].
//
// Replaces the model's own attention where the reference calls it for a
// query of many positions: every prefill chunk (kiv/middleware.py:174-260
// runs the original attention there) and a multi-position query over
// [retrieved ; hot] (kiv/middleware.py:343-352).  Semantics of the eager
// reference (third-party modeling_qwen2.py:150-172): scores * scaling +
// mask, softmax in fp32, probabilities rounded to the activation dtype,
// then @ V.  Here the probabilities are rounded before the normalisation
// (flash style), which moves each output by at most the probabilities'
// own rounding, u * sum_k p_k |v_k|.
//
// Blocks of 256 threads own 128 query rows of one q head (64 above head_dim
// 128).  Keys come in tiles of 64: first the retrieved keys, then the hot
// keys (a tile never mixes the two, so hot tiles line up with the mask's
// column tiles).  Online softmax in base 2; the running maximum is raised,
// and the accumulators rescaled, only when a score exceeds it by more than
// 2^8, so probabilities stay below 256 and most tiles skip the rescale and
// the cross-lane maxima.
//
// Head dims up to 128 (prefill_attn32_kernel, below): 32 query rows a wave,
// the work dealt to the GPU's block slots in equal shares (PfShares).  The
// model's chunk, 4096 x 8192 keys of 12 heads under a boolean mask: 230 ->
// 181 to 189 us a call by the box, 155 GFLOP; the attention kernel's matrix
// cores are busy 41% of its cycles (28% before), bound by the issue of the
// softmax beside the matrix instructions with two waves a SIMD.
//
// Head dims above 128 (prefill_attn_kernel): wave w holds 16 query rows.
// The grid is one-dimensional in longest-first order and long rows are split
// over key ranges whose partial rows a combine kernel merges.  Per tile:
//  - K rows ([64][D], rows padded by 16 bytes) and V transposed ([D][64],
//    rows padded by 8 bytes) go to LDS from registers that were loaded
//    (buffer loads bounded to the segment) while the previous tile was
//    being computed;
//  - S^T = K Q^T with v_mfma_f32_16x16x32: lane l gives row l % 16 of a
//    16-key sub-tile of K (A) and its own query row l % 16 (B, held in
//    registers for the whole kernel), dims 32 s + 8 (l / 16) .. + 7 of
//    step s, and receives keys 4 (l / 16) + i of the sub-tile for its row;
//  - O^T += V^T P^T with v_mfma_f32_16x16x32 over 32 keys: the B operand is
//    exactly the lane's probabilities of two sub-tiles (k index 8 g + i is
//    key 4 g + i of the first sub-tile for i < 4, of the second for i >= 4),
//    the A operand the same keys of one dim from the V^T tile.  All O^T
//    entries of a lane belong to its query row.
//
// Tile classes: SKIP (no row of the block sees a key of the tile), FULL
// (every key present and visible with zero bias: no per-element work) and
// MIXED.  The causal rule and the tile edges give them arithmetically; for
// a mask tensor a first kernel classifies every (mask row block, column
// tile) once, so the attention reads mask elements only in MIXED tiles.
#include <algorithm>
#include <climits>

#include "kiv_common.h"
#include "kiv_dispatch.h"
#include "kiv_internal.h"
#include "kiv_prefill_shares.h"

namespace kiv {

constexpr int kPfThreads = 256;
constexpr int kPfRows = 64;  // query rows per mask tile class entry
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kRescaleSlack = 8.f;  // base-2 headroom before the running max moves
enum { TILE_SKIP = 0, TILE_FULL = 1, TILE_MIXED = 2 };
enum { PF_ARITH = 0, PF_BOOL = 1, PF_FLOAT = 2 };  // how MIXED tiles get their bias

struct PrefillParams {
  const char *q;
  int64_t qs0, qs1, qs2;
  const char *cold_k, *cold_v;
  int cold_len, hot_len;
  const char *hot_k, *hot_v;
  int64_t hks0, hks1, hks2, hvs0, hvs1, hvs2;
  const char *mask;
  int mask_kind;  // KIV_MASK_*
  int mask_vec4;  // bool mask with 4-byte aligned rows of unit stride
  int64_t ms0, ms1, ms2, ms3;
  uint8_t *tiles;  // [Bm][Hm][ceil(Q/64)][ceil(T/64)] TILE_* of the hot columns
  int mask_b, mask_h;    // Bm, Hm: 1 where the mask broadcasts
  int batch, hq, hkv, qlen;
  float scale_log2;  // scaling * log2(e)
  char *out;
  // Key splits (head dims above 128): with nsplit > 1 each split writes its unnormalised
  // rows and (running max, row sum) here and prefill_combine_kernel merges.
  int nsplit;
  float *ws_m, *ws_l, *ws_o;  // [nsplit][B*Q*Hq], [nsplit][B*Q*Hq], [nsplit][B*Q*Hq][D]
  PfShares sh;                // head dims up to 128: the blocks' shares (then ws_* are [2 * blocks][part_rows])
  int part_rows;
  int2 *cuts;  // with shares, per unit: 2 * its first block + (not that block's first fragment), its last block
  // Mask tensors under shares: a bit per hot tile that a 64-row entry sees,
  // [Bm][Hm][2 * row blocks][1 << seen_shift] words, zero past the last tile
  // and row.
  uint32_t *seen;
  int seen_shift;
};

// N bytes at p, of any alignment (mask rows start anywhere: a hot window of
// T columns puts consecutive rows T elements apart); the compiler emits one
// vector load where the target allows it.
template <typename T> __device__ __forceinline__ T load_any(const char *p) {
  T v;
  __builtin_memcpy(&v, p, sizeof(T));
  return v;
}
// Four consecutive float-mask elements from element o on (base 2).
__device__ __forceinline__ void float_bias4(const PrefillParams &p, int64_t o, float (&bias)[4]) {
  if (p.mask_kind == KIV_MASK_F32) {
    const uint4 v = load_any<uint4>(p.mask + 4 * o);
    bias[0] = __uint_as_float(v.x) * kLog2e;
    bias[1] = __uint_as_float(v.y) * kLog2e;
    bias[2] = __uint_as_float(v.z) * kLog2e;
    bias[3] = __uint_as_float(v.w) * kLog2e;
    return;
  }
  const uint2 v = load_any<uint2>(p.mask + 2 * o);
  const uint32_t w[4] = {v.x & 0xffffu, v.x >> 16, v.y & 0xffffu, v.y >> 16};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    bias[i] = (p.mask_kind == KIV_MASK_F16 ? f16_bits_to_f32(w[i]) : bf16_bits_to_f32(w[i])) * kLog2e;
}

// Two fp32 values rounded to the dtype (hardware conversion, nearest even),
// packed low-first.
template <int DT> __device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (DT == DT_BF16) return __builtin_bit_cast(uint32_t, bf16x2_t{(__bf16)a, (__bf16)b});
  else return __builtin_bit_cast(uint32_t, f16x2_t{(_Float16)a, (_Float16)b});
}

__device__ __forceinline__ int64_t mask_off(const PrefillParams &p, int b, int h, int i, int t) {
  return (int64_t)b * p.ms0 + (int64_t)h * p.ms1 + (int64_t)i * p.ms2 + (int64_t)t * p.ms3;
}

// Additive bias (base 2) of a float mask element.
__device__ __forceinline__ float float_bias(const PrefillParams &p, int64_t o) {
  switch (p.mask_kind) {
    case KIV_MASK_F32: return load_elem<DT_F32>(p.mask, o) * kLog2e;
    case KIV_MASK_F16: return load_elem<DT_F16>(p.mask, o) * kLog2e;
    default: return load_elem<DT_BF16>(p.mask, o) * kLog2e;
  }
}

// Query rows per block: 32 a wave up to head_dim 128 (each K and V^T operand
// read from LDS then feeds a 32x32 matrix instruction), 16 above (the
// accumulators would not fit).
template <int KT> struct PfShape {
  static constexpr int ROWS = KT <= 4 ? 128 : 64;
};
constexpr int kPfLdsTiles = 4096;  // tile classes a block keeps in LDS (hot windows up to 256K keys)

// One block's share of the work: its query rows, its key tiles and their
// classes, and the staging of K and V tiles through registers into LDS (K
// rows [64][D] padded by 16 bytes, V transposed [D][64] padded by 8 bytes).
template <int DT, int KT, int MK> struct PfGeom {
  static constexpr int D = 32 * KT, CPR = D / 8, NT = kPfThreads, ROWS = PfShape<KT>::ROWS;
  static_assert(ROWS % 64 == 0, "a block covers whole 64-row mask class entries");

  const PrefillParams &p;
  int b, h, kvh, z, tid, wave, lane, q0, qlast, off, nct, nht, t_begin, t_end;
  bool causal;
  const uint8_t *cls_rows;
  int cls_n;
  const char *cold_kb, *cold_vb, *hot_kb, *hot_vb;

  __device__ __forceinline__ explicit PfGeom(const PrefillParams &pp) : p(pp) {
    z = 0;
    tid = threadIdx.x;
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    lane = tid & 63;
    off = p.hot_len - p.qlen;  // causal: hot column t visible to row i iff t <= i + off
    causal = p.mask_kind == KIV_MASK_CAUSAL;
    nct = (p.cold_len + kPfKeys - 1) / kPfKeys;
    nht = (p.hot_len + kPfKeys - 1) / kPfKeys;
  }

  // Row block rb of (b, q head) bh, its tiles [t0, t1).
  __device__ __forceinline__ void set_unit(int bh, int rb, int t0, int t1) {
    b = bh / p.hq;
    h = bh - b * p.hq;
    kvh = h / (p.hq / p.hkv);
    q0 = rb * ROWS;
    qlast = min(q0 + ROWS, p.qlen) - 1;
    t_begin = t0;
    t_end = t1;
    // Mask tensors: the classes of this block's rows (the 64-row entries it
    // spans, to be combined).
    cls_rows = nullptr;
    cls_n = 0;
    if constexpr (MK != PF_ARITH) {
      const int mb = p.mask_b == 1 ? 0 : b, mh = p.mask_h == 1 ? 0 : h;
      const int nqb = (p.qlen + 63) / 64, r0 = q0 / 64;
      const int64_t entry = (int64_t)(mb * p.mask_h + mh) * nqb + r0;
      cls_n = min(ROWS / 64, nqb - r0);
      cls_rows = p.tiles + entry * nht;
    }
    cold_kb = p.cold_k + ((int64_t)b * p.hkv + kvh) * p.cold_len * (int64_t)D * 2;
    cold_vb = p.cold_v + ((int64_t)b * p.hkv + kvh) * p.cold_len * (int64_t)D * 2;
    hot_kb = p.hot_k + ((int64_t)b * p.hks0 + (int64_t)kvh * p.hks1) * 2;
    hot_vb = p.hot_v + ((int64_t)b * p.hvs0 + (int64_t)kvh * p.hvs1) * 2;
  }

  __device__ __forceinline__ int combine(int k) const {
    int c = cls_rows[k];
    for (int r = 1; r < cls_n; ++r) {
      const int d = cls_rows[(int64_t)r * nht + k];
      c = c == d ? c : (c == TILE_SKIP && d == TILE_SKIP) ? TILE_SKIP : TILE_MIXED;
    }
    return c;
  }
  // Class of tile t for this block (mask tensors: read from memory).
  __device__ __forceinline__ int tile_class_of(int t) const {
    if (t < nct) return (t + 1) * kPfKeys <= p.cold_len ? TILE_FULL : TILE_MIXED;
    if constexpr (MK == PF_ARITH) {
      const int key0 = (t - nct) * kPfKeys;
      const bool whole = key0 + kPfKeys <= p.hot_len;
      if (!causal) return whole ? TILE_FULL : TILE_MIXED;
      if (key0 > qlast + off) return TILE_SKIP;
      return whole && key0 + kPfKeys - 1 <= q0 + off ? TILE_FULL : TILE_MIXED;
    } else {
      return combine(t - nct);
    }
  }

  // Bias of four consecutive keys k4 .. k4 + 3 of a MIXED tile (its first
  // key key0 of its segment, n keys left in it) for query row qrow, whose
  // mask offset is row_mo: 0 or -inf, or the float mask's value (base 2).
  __device__ __forceinline__ void bias4(bool cold, int key0, int n, int k4, int qrow, int64_t row_mo,
                                        float (&bias)[4]) const {
    const int64_t mo = row_mo + (int64_t)(key0 + k4) * p.ms3;
    if (cold || MK == PF_ARITH) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool vis = k4 + i < n && (cold || !causal || key0 + k4 + i <= qrow + off);
        bias[i] = vis ? 0.f : -INFINITY;
      }
    } else if (MK == PF_BOOL) {
      uint32_t bits = 0;
      if (p.mask_vec4 && k4 + 4 <= n) {
        bits = *reinterpret_cast<const uint32_t *>(p.mask + mo);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (k4 + i < n && p.mask[mo + (int64_t)i * p.ms3]) bits |= 0xffu << (8 * i);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) bias[i] = (bits >> (8 * i)) & 0xffu ? 0.f : -INFINITY;
    } else if (p.ms3 == 1 && n >= kPfKeys) {
      float_bias4(p, mo, bias);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) bias[i] = k4 + i < n ? float_bias(p, mo + (int64_t)i * p.ms3) : -INFINITY;
    }
  }
  __device__ __forceinline__ int64_t row_mask_off(int qrow) const { return mask_off(p, b, h, qrow, 0); }

  // Four consecutive output dims d .. d + 3 of query row qrow: normalised,
  // or (with key splits) this split's unnormalised sums.
  __device__ __forceinline__ int64_t split_row(int qrow) const {
    return (int64_t)z * p.batch * p.qlen * p.hq + ((int64_t)b * p.qlen + qrow) * p.hq + h;
  }
  __device__ __forceinline__ char *out_row(int qrow) const {
    return p.out + (((int64_t)b * p.qlen + qrow) * p.hq + h) * (int64_t)D * 2;
  }
};

// Head dims above 128: a wave holds 16 query rows, tiles go to LDS through
// registers (K rows padded by 16 bytes, V transposed).
template <int DT, int KT, int MK> struct PfBlock : PfGeom<DT, KT, MK> {
  using Geom = PfGeom<DT, KT, MK>;
  using Geom::b, Geom::CPR, Geom::cold_kb, Geom::cold_vb, Geom::D, Geom::h, Geom::hot_kb, Geom::hot_vb, Geom::NT,
      Geom::nct, Geom::p, Geom::t_begin, Geom::t_end, Geom::tid, Geom::wave, Geom::lane, Geom::q0, Geom::z;
  static constexpr int KROW = D + 8;        // K tile row stride in elements
  static constexpr int VROW = kPfKeys + 4;  // V^T tile row stride in elements
  static constexpr int KTILE = kPfKeys * KROW, VTILE = D * VROW;  // elements of one LDS tile
  static constexpr int KJ = (kPfKeys * CPR + NT - 1) / NT;          // K chunks per thread
  static constexpr int VJ = ((kPfKeys / 4) * CPR + NT - 1) / NT;    // V key quads per thread
  const uint8_t *tcls;  // LDS copy of this block's hot tile classes (mask tensors)
  bool cls_lds;
  int col, grp;
  int qi, qc;  // the lane's query row (rows past Q repeat row Q - 1's data)
  uint4 kreg[KJ], vreg[VJ][4];

  // Class of tile t, uniform over the block.
  __device__ __forceinline__ int tile_class(int t) const {
    if (MK == PF_ARITH || t < nct) return this->tile_class_of(t);
    return __builtin_amdgcn_readfirstlane(cls_lds ? (int)tcls[t - nct] : this->combine(t - nct));
  }
  // The first tile after t that is not skipped, or t_end.
  __device__ __forceinline__ int next_tile(int t) const {
    for (++t; t < t_end; ++t) {
      if constexpr (MK == PF_ARITH) {
        // The causal rule hides every tile after the first hidden one.
        if (this->causal && t >= nct && (t - nct) * kPfKeys > this->qlast + this->off) return t_end;
      }
      if (tile_class(t) != TILE_SKIP) return t;
    }
    return t_end;
  }
  __device__ __forceinline__ int first_tile() const {
    return t_begin < t_end && tile_class(t_begin) != TILE_SKIP ? t_begin : next_tile(t_begin);
  }

  __device__ __forceinline__ PfBlock(const PrefillParams &pp, uint8_t *tcls_lds) : Geom(pp), tcls(tcls_lds) {
    // One-dimensional grid, longest work first: row blocks from the last
    // (under the causal rule later rows see more tiles), then batch rows,
    // heads and key splits, so that the dispatcher hands out the block
    // slots longest-first and the launch ends with short blocks.
    const int per_rb = p.batch * p.hq * p.nsplit, lin = blockIdx.x;
    const int nrb = gridDim.x / per_rb, rb = lin / per_rb, rem = lin - rb * per_rb;
    const int bh = rem / p.nsplit;
    z = rem - bh * p.nsplit;
    // This block's share of the tiles (all of them without key splits).
    const int ntiles = nct + this->nht;
    this->set_unit(bh, nrb - 1 - rb, (int)((int64_t)z * ntiles / p.nsplit), (int)((int64_t)(z + 1) * ntiles / p.nsplit));
    cls_lds = MK != PF_ARITH && this->nht <= kPfLdsTiles;
    if (cls_lds) {
      for (int k = tid; k < this->nht; k += NT) tcls_lds[k] = (uint8_t)this->combine(k);
      __syncthreads();
    }
    col = lane & 15;
    grp = lane >> 4;
    qi = q0 + 16 * wave + col;
    qc = min(qi, p.qlen - 1);
  }

  // Loads tile t's K chunks (V key quads) into registers through a buffer
  // that ends at the segment's last row: rows past it read as zeros, and
  // their scores get a -inf bias (a tile that is not whole is MIXED).
  __device__ __forceinline__ void load_k(int t) {
    const bool cold = t < nct;
    const int key0 = (cold ? t : t - nct) * kPfKeys, rows = min(kPfKeys, (cold ? p.cold_len : p.hot_len) - key0);
    const uint32_t krs = cold ? D * 2 : (uint32_t)p.hks2 * 2;
    const auto rk = tile_rsrc((cold ? cold_kb : hot_kb) + (int64_t)key0 * krs, (uint32_t)rows * krs);
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      const int i = tid + j * NT, key = i / CPR, c = i - key * CPR;
      kreg[j] = buf_load16(rk, (uint32_t)key * krs + c * 16);
    }
  }
  __device__ __forceinline__ void load_v(int t) {
    const bool cold = t < nct;
    const int key0 = (cold ? t : t - nct) * kPfKeys, rows = min(kPfKeys, (cold ? p.cold_len : p.hot_len) - key0);
    const uint32_t vrs = cold ? D * 2 : (uint32_t)p.hvs2 * 2;
    const auto rv = tile_rsrc((cold ? cold_vb : hot_vb) + (int64_t)key0 * vrs, (uint32_t)rows * vrs);
#pragma unroll
    for (int j = 0; j < VJ; ++j) {
      const int i = tid + j * NT, quad = i % (kPfKeys / 4), c = i / (kPfKeys / 4);
      if (VJ * NT == (kPfKeys / 4) * CPR || i < (kPfKeys / 4) * CPR) {
        const uint32_t voff = (uint32_t)(4 * quad) * vrs + c * 16;
#pragma unroll
        for (int r = 0; r < 4; ++r) vreg[j][r] = buf_load16(rv, voff + (uint32_t)r * vrs);
      }
    }
  }
  __device__ __forceinline__ void store_k(uint16_t *ks) const {
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      const int i = tid + j * NT, key = i / CPR, c = i - key * CPR;
      *reinterpret_cast<uint4 *>(&ks[key * KROW + c * 8]) = kreg[j];
    }
  }
  __device__ __forceinline__ void store_v(uint16_t *vt) const {
#pragma unroll
    for (int j = 0; j < VJ; ++j) {
      const int i = tid + j * NT, quad = i % (kPfKeys / 4), c = i / (kPfKeys / 4);
      if (VJ * NT == (kPfKeys / 4) * CPR || i < (kPfKeys / 4) * CPR) {
        const uint32_t w[4][4] = {{vreg[j][0].x, vreg[j][0].y, vreg[j][0].z, vreg[j][0].w},
                                  {vreg[j][1].x, vreg[j][1].y, vreg[j][1].z, vreg[j][1].w},
                                  {vreg[j][2].x, vreg[j][2].y, vreg[j][2].z, vreg[j][2].w},
                                  {vreg[j][3].x, vreg[j][3].y, vreg[j][3].z, vreg[j][3].w}};
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          // dims 2m (low halves) and 2m + 1 (high halves) of the four keys,
          // one byte permute per pair (bytes 0-3 of the selector's table are
          // the second operand, 4-7 the first)
          const uint2 lo = make_uint2(__builtin_amdgcn_perm(w[1][m], w[0][m], 0x05040100u),
                                      __builtin_amdgcn_perm(w[3][m], w[2][m], 0x05040100u));
          const uint2 hi = make_uint2(__builtin_amdgcn_perm(w[1][m], w[0][m], 0x07060302u),
                                      __builtin_amdgcn_perm(w[3][m], w[2][m], 0x07060302u));
          *reinterpret_cast<uint2 *>(&vt[(c * 8 + 2 * m) * VROW + 4 * quad]) = lo;
          *reinterpret_cast<uint2 *>(&vt[(c * 8 + 2 * m + 1) * VROW + 4 * quad]) = hi;
        }
      }
    }
  }

  // The lane's query fragments: row qc, dims 32 st + 8 grp .. + 7 of step st.
  __device__ __forceinline__ void load_q(uint4 (&qx)[KT]) const {
    const char *qrow = p.q + ((int64_t)b * p.qs0 + (int64_t)h * p.qs1 + (int64_t)qc * p.qs2) * 2;
#pragma unroll
    for (int st = 0; st < KT; ++st) qx[st] = load16(qrow + (32 * st + 8 * grp) * 2);
  }

  // MIXED tile t: scores become s * scaling * log2 e + bias (base 2), so the
  // tile's remaining factor is 1.
  __device__ __forceinline__ void add_bias(f32x4_t (&s)[4], int t) const {
    const bool cold = t < nct;
    const int key0 = (cold ? t : t - nct) * kPfKeys, n = (cold ? p.cold_len : p.hot_len) - key0;
    const int64_t row_mo = this->row_mask_off(qc);
#pragma unroll
    for (int sub = 0; sub < 4; ++sub) {
      float bias[4];
      this->bias4(cold, key0, n, 16 * sub + 4 * grp, qc, row_mo, bias);
#pragma unroll
      for (int i = 0; i < 4; ++i) s[sub][i] = fmaf(s[sub][i], p.scale_log2, bias[i]);
    }
  }

  // The block's rows: normalised output, or (with key splits) this split's
  // unnormalised rows with their running max and row sum.
  __device__ __forceinline__ void finish(const f32x4_t (&o)[D / 16], float m_run, float l_lane) const {
    const float l_row = half_wave_sum(row_pair_sum(l_lane));
    if (qi >= p.qlen) return;
    if (p.nsplit > 1) {
      const int64_t sr = this->split_row(qi);
      float *po = p.ws_o + sr * D;
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt) *reinterpret_cast<f32x4_t *>(po + 16 * dt + 4 * grp) = o[dt];
      if (grp == 0) {
        p.ws_m[sr] = m_run;
        p.ws_l[sr] = l_row;
      }
      return;
    }
    // A row with no visible key (fully masked) gets zeros.
    const float inv = l_row > 0.f ? 1.f / l_row : 0.f;
    char *orow = this->out_row(qi);
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt)
      *reinterpret_cast<uint2 *>(orow + (16 * dt + 4 * grp) * 2) =
          make_uint2(pack2<DT>(o[dt][0] * inv, o[dt][1] * inv), pack2<DT>(o[dt][2] * inv, o[dt][3] * inv));
  }
};

// S^T = K Q^T for one tile with v_mfma_f32_16x16x32: lane l gives row l % 16
// of a 16-key sub-tile of K (A) and its own query row l % 16 (B), dims
// 32 st + 8 (l / 16) .. + 7 of step st, and receives keys 4 (l / 16) + i of
// the sub-tile for its row.
template <int DT, int KT>
__device__ __forceinline__ void pf_scores(f32x4_t (&s)[4], const uint16_t *ks, const uint4 (&qx)[KT], int col,
                                          int grp) {
  constexpr int KROW = 32 * KT + 8;
#pragma unroll
  for (int sub = 0; sub < 4; ++sub) s[sub] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int st = 0; st < KT; ++st)
#pragma unroll
    for (int sub = 0; sub < 4; ++sub) {
      const uint4 a = *reinterpret_cast<const uint4 *>(&ks[(16 * sub + col) * KROW + 32 * st + 8 * grp]);
      s[sub] = mfma_16x16x32<DT>(a, qx[st], s[sub]);
    }
}

// Raises a row's running max (and rescales its accumulators) only when the
// tile's max is more than 2^kRescaleSlack above it, so probabilities stay
// below 256 and most tiles skip the rescale; the wave skips it when no lane
// needs it.  Each lane's own maximum, over its 16 scores, is tested first: the
// maximum of a row exceeds the bound exactly when that of one of its four
// lanes (l, l ^ 16, l ^ 32, l ^ 48) does (the scale cc > 0 and its rounding
// are monotone), so the rows' maxima across lanes are only formed on the tiles
// that raise one.
template <int NO>
__device__ __forceinline__ void pf_max_raise(const f32x4_t (&s)[4], float cc, float &m_run, float &l_lane,
                                             f32x4_t (&o)[NO]) {
  float x = s[0][0];
#pragma unroll
  for (int sub = 0; sub < 4; ++sub)
#pragma unroll
    for (int i = 0; i < 4; ++i) x = fmaxf(x, s[sub][i]);
  if (!__ballot(x * cc > m_run + kRescaleSlack)) return;
  const float mt = half_wave_max(row_pair_max(x)) * cc;
  const float m_new = mt > m_run + kRescaleSlack ? mt : m_run;
  const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
  l_lane *= alpha;
#pragma unroll
  for (int dt = 0; dt < NO; ++dt) o[dt] *= alpha;
  m_run = m_new;
}

// Probabilities of one tile, 2^(cc s - m) rounded to the dtype and packed as
// the B operand of O^T += V^T P^T: k index 8 g + i of pb[j] is key
// 4 g + i of sub-tile 2 j for i < 4, of sub-tile 2 j + 1 for i >= 4.  The
// lane's share of each row sum grows by their fp32 values.  A row that has
// seen no key keeps m = -inf; its probabilities are 0.
template <int DT>
__device__ __forceinline__ void pf_probs(const f32x4_t (&s)[4], float cc, float m_run, float &l_lane,
                                         uint4 (&pb)[2]) {
  const float m_neg = m_run == -INFINITY ? 0.f : -m_run;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float e[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      e[i] = __builtin_amdgcn_exp2f(fmaf(s[2 * j][i], cc, m_neg));
      e[4 + i] = __builtin_amdgcn_exp2f(fmaf(s[2 * j + 1][i], cc, m_neg));
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) l_lane += e[i];
    pb[j] = make_uint4(pack2<DT>(e[0], e[1]), pack2<DT>(e[2], e[3]), pack2<DT>(e[4], e[5]), pack2<DT>(e[6], e[7]));
  }
}

// O^T += V^T P^T with v_mfma_f32_16x16x32 over 32 keys at a time: the A
// operand holds the same keys of one dim from the V^T tile; every O^T entry
// of a lane belongs to its query row.
template <int DT, int D>
__device__ __forceinline__ void pf_pv(f32x4_t (&o)[D / 16], const uint4 (&pb)[2], const uint16_t *vt, int col,
                                      int grp) {
  constexpr int VROW = kPfKeys + 4;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) {
      const uint16_t *vr = &vt[(16 * dt + col) * VROW + 32 * j + 4 * grp];
      const uint2 lo = *reinterpret_cast<const uint2 *>(vr), hi = *reinterpret_cast<const uint2 *>(vr + 16);
      const uint4 a = make_uint4(lo.x, lo.y, hi.x, hi.y);
      o[dt] = mfma_16x16x32<DT>(a, pb[j], o[dt]);
    }
}

// ---------------------------------------------------------------------------
// Tile classes of a mask tensor: grid (column tile groups, row blocks,
// Bm * Hm), 256 threads; a block classifies kMaskTilesPerBlock consecutive
// 64 x 64 tiles of one row block (its loads all in flight together), thread
// t covering row q0 + t / 4, columns 16 (t % 4) .. + 15 of each.  Rows past
// Q do not count; columns past T make a tile MIXED.
constexpr int kMaskTilesPerBlock = 8;
__global__ void __launch_bounds__(kPfThreads) mask_tiles_kernel(PrefillParams p) {
  constexpr int TPB = kMaskTilesPerBlock, W = kPfThreads / 64;
  __shared__ uint8_t wany[TPB][W], wall[TPB][W];
  const int qb = blockIdx.y, bh = blockIdx.z, tid = threadIdx.x, wave = tid >> 6;
  const int mb = bh / p.mask_h, mh = bh - mb * p.mask_h;
  const int nkt = (p.hot_len + kPfKeys - 1) / kPfKeys, kt0 = blockIdx.x * TPB;
  const int row = qb * kPfRows + (tid >> 2), cq = 16 * (tid & 3);
  int any[TPB], all[TPB];
#pragma unroll
  for (int j = 0; j < TPB; ++j) {
    any[j] = 0;
    all[j] = 1;
  }
  // Columns c0 .. c0 + 15 of one tile into any / all.
  auto scalar = [&](int64_t o, int c0, int &an, int &al) {
    for (int e = 0; e < 16; ++e) {
      const int t = c0 + e;
      if (t >= p.hot_len) {
        al = 0;
        continue;
      }
      const int64_t oe = o + (int64_t)t * p.ms3;
      if (p.mask_kind == KIV_MASK_BOOL) {
        const bool vis = p.mask[oe] != 0;
        an |= vis;
        al &= vis;
      } else {
        const float v = float_bias(p, oe);
        an |= v != -INFINITY;
        al &= v == 0.f;
      }
    }
  };
  if (row < p.qlen) {
    const int64_t o = mask_off(p, mb, mh, row, 0);
    if (p.mask_kind == KIV_MASK_BOOL && p.ms3 == 1) {
      uint4 v[TPB];
#pragma unroll
      for (int j = 0; j < TPB; ++j) {
        const int c0 = (kt0 + j) * kPfKeys + cq;
        v[j] = c0 + 16 <= p.hot_len ? load_any<uint4>(p.mask + o + c0) : make_uint4(0, 0, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < TPB; ++j) {
        const int c0 = (kt0 + j) * kPfKeys + cq;
        if (kt0 + j >= nkt) continue;
        if (c0 + 16 <= p.hot_len) {
          const uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const bool vis = (w[q] >> (8 * e)) & 0xffu;
              any[j] |= vis;
              all[j] &= vis;
            }
        } else {
          scalar(o, c0, any[j], all[j]);
        }
      }
    } else if (p.mask_kind != KIV_MASK_BOOL && p.ms3 == 1) {
#pragma unroll
      for (int j = 0; j < TPB; ++j) {
        const int c0 = (kt0 + j) * kPfKeys + cq;
        if (kt0 + j >= nkt) continue;
        if (c0 + 16 <= p.hot_len) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            float v[4];
            float_bias4(p, o + c0 + 4 * u, v);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              any[j] |= v[e] != -INFINITY;
              all[j] &= v[e] == 0.f;
            }
          }
        } else {
          scalar(o, c0, any[j], all[j]);
        }
      }
    } else {
      for (int j = 0; j < TPB && kt0 + j < nkt; ++j) scalar(o, (kt0 + j) * kPfKeys + cq, any[j], all[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < TPB; ++j) {
    const uint64_t a = __ballot(any[j]), n = __ballot(!all[j]);
    if ((tid & 63) == 0) {
      wany[j][wave] = a != 0;
      wall[j][wave] = n == 0;
    }
  }
  __syncthreads();
  if (wave != 0) return;
  const int nqb = (p.qlen + kPfRows - 1) / kPfRows;
  const int64_t entry = (int64_t)bh * nqb + qb;
  int an = 0, al = 1;
  if (tid < TPB && kt0 + tid < nkt) {
#pragma unroll
    for (int w = 0; w < W; ++w) {
      an |= wany[tid][w];
      al &= wall[tid][w];
    }
    p.tiles[entry * nkt + kt0 + tid] = (uint8_t)(!an ? TILE_SKIP : al ? TILE_FULL : TILE_MIXED);
  }
  if (p.seen) {
    // This block's byte of the row's bits; the last blocks also write the
    // zeros after the row and a missing second row of the row block.
    static_assert(TPB == 8, "a block's tiles are one byte of bits");
    const uint64_t seen = __ballot(an);
    const int bytes = 4 << p.seen_shift, last = blockIdx.x == gridDim.x - 1 ? bytes : (int)blockIdx.x + 1;
    uint8_t *row = reinterpret_cast<uint8_t *>(p.seen) + ((int64_t)bh * 2 * p.sh.nrb + qb) * bytes;
    for (int at = (int)blockIdx.x + tid; at < last; at += 64) {
      row[at] = at == (int)blockIdx.x ? (uint8_t)seen : 0;
      if (qb == nqb - 1 && !(qb & 1)) row[bytes + at] = 0;
    }
  }
}

// ---------------------------------------------------------------------------
// Head dims up to 128: 32 query rows a wave on v_mfma_f32_32x32x16.
//
// K and V tiles go from memory straight to LDS (buffer loads of 16 bytes a
// lane into 1 KiB of LDS an instruction), both as rows, double-buffered: a
// tile has the whole computation of the one before it to arrive, and a wave
// passes one barrier a tile.  LDS rows hold CP 16-byte chunks (head_dim 96
// is padded to 16 chunks); the chunks of a row are permuted so that every
// operand read spreads over the banks (K by row, so that 16 rows' same chunk
// lie in 16 different places; V by key, so that four keys' 64-byte pieces
// do), which the loading lanes do by fetching the permuted chunk.
//  - S^T = K Q^T: lane l gives row l % 32 of a 32-key sub-tile of K (A) and
//    its own query row l % 32 (B, in registers for the whole kernel), dims
//    16 st + 8 (l / 32) .. + 7 of step st, and receives keys
//    8 (i / 4) + 4 (l / 32) + i % 4 (i < 16) of the sub-tile for its row.
//  - O^T += V^T P^T, 16 keys a step: the B operand is the lane's own
//    probabilities 8 j .. 8 j + 7 of a sub-tile (keys 16 j + 4 (l / 32) + i
//    for i < 4, 16 j + 8 + 4 (l / 32) + i - 4 for i >= 4), the A operand the
//    same keys of dim l % 32, from two transposing LDS reads
//    (ds_read_b64_tr_b16: each 16 lanes read 4 keys x 16 dims and lane n
//    receives the 4 keys of dim n).
typedef float f32x16_t __attribute__((ext_vector_type(16)));
template <int DT> __device__ __forceinline__ f32x16_t mfma_32x32x16(const uint4 &a, const uint4 &b, f32x16_t c) {
  if constexpr (DT == DT_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                    c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                   0, 0, 0);
}
constexpr int kWaitMem = 0x0070;  // s_waitcnt vmcnt(0) lgkmcnt(0)
typedef __attribute__((address_space(3))) void lds_void_t;
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4_t lds_i16x4_t;

template <int DT, int KT, int MK> struct PfBlock32 : PfGeom<DT, KT, MK> {
  using Geom = PfGeom<DT, KT, MK>;
  using Geom::b, Geom::CPR, Geom::cold_kb, Geom::cold_vb, Geom::D, Geom::h, Geom::hot_kb, Geom::hot_vb, Geom::nct,
      Geom::p, Geom::t_begin, Geom::t_end, Geom::wave, Geom::lane, Geom::q0;
  static constexpr int CP = CPR <= 4 ? 4 : CPR <= 8 ? 8 : 16;  // chunks per LDS row
  static constexpr int RPI = 64 / CP;                          // rows per load instruction
  static constexpr int NJ = CP / 4;                            // load instructions per wave for a tile of K (of V)
  static constexpr int TILE = kPfKeys * CP * 8;                // elements of a tile in LDS
  static constexpr int KS = D / 16, ND = D / 32;               // score steps, output dim tiles
  int row, hf;         // the lane's query row (column of both products) and half
  int qi, qc;          // its query position; the last one for rows past Q
  int lrow, kc, vc;    // loads: the lane's row of the wave's first instruction, its K and V chunk bytes
  int kaddr, vaddr[ND];  // operand reads: byte offsets of the lane within a K / V tile

  int wbase;             // tiles wbase .. + 63 as bits: not skipped, and mixed
  uint64_t wseen, wmixed;

  __device__ __forceinline__ explicit PfBlock32(const PrefillParams &pp) : Geom(pp) {
    row = lane & 31;
    hf = lane >> 5;
    // Row r holds K chunk c at c ^ xk(r), xk(r) = r / (16 / CP) mod CP, and
    // V chunk c at c ^ 4 xv(r), xv(r) = r mod 4 (16 chunks) or r / 2 mod 2
    // (8) or 0 (4): the same for every load instruction of a lane, whose
    // rows are 4 RPI apart.
    lrow = wave * RPI + lane / CP;
    const int pc = lane % CP;
    kc = min(pc ^ ((lrow / (16 / CP)) & (CP - 1)), CPR - 1) * 16;
    vc = min(pc ^ (4 * xv(lrow)), CPR - 1) * 16;
    kaddr = row * CP * 16 + ((hf ^ ((row / (16 / CP)) & (CP - 1))) << 4);
    const int j16 = lane & 15, q = j16 >> 2;  // the transposing read: key q of four, dims 4 (j16 % 4) ..
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) {
      const int c = 4 * (dt ^ xv(q)) + 2 * ((lane >> 4) & 1) + ((j16 & 3) >> 1);
      vaddr[dt] = (4 * hf + q) * CP * 16 + c * 16 + (j16 & 1) * 8;
    }
  }
  __device__ __forceinline__ void set_unit(int bh, int rb, int t0, int t1) {
    Geom::set_unit(bh, rb, t0, t1);
    qi = q0 + 32 * wave + row;
    qc = min(qi, p.qlen - 1);
  }
  // The classes of 64 tiles in scalar registers, a tile a lane: the loop
  // finds its next tile with scalar bit operations.
  __device__ __forceinline__ void window(int base) {
    wbase = base;
    const int t = base + lane, cls = t < t_end ? this->tile_class_of(t) : (int)TILE_SKIP;
    wseen = __ballot(cls != TILE_SKIP);
    wmixed = __ballot(cls == TILE_MIXED);
  }
  // Mask tensors: word base + lane of the unit's bits of visible hot tiles.
  __device__ __forceinline__ uint32_t seen_bits(int base) const {
    const int mb = p.mask_b == 1 ? 0 : b, mh = p.mask_h == 1 ? 0 : h, at = base + lane;
    const uint32_t *row =
        p.seen + (((int64_t)(mb * p.mask_h + mh) * p.sh.nrb * 2 + q0 / 64) << p.seen_shift) + at;
    return at < 1 << p.seen_shift ? row[0] | row[1 << p.seen_shift] : 0u;
  }
  // The tile that v visible tiles of the unit precede (the retrieved keys'
  // tiles are all visible), or all tiles past the last; bits: seen_bits(0).
  __device__ __forceinline__ int locate(int v, uint32_t bits) const {
    if (v < nct) return v;
    v -= nct;
    for (int base = 0; base < 1 << p.seen_shift; base += 64) {
      if (base > 0) bits = seen_bits(base);
      const int upto = wave_incl_scan(__popc(bits));  // visible tiles up to this lane's word
      const uint64_t past = __ballot(upto > v);
      if (past) {
        const int l = __builtin_ctzll(past);
        uint32_t word = (uint32_t)__builtin_amdgcn_readlane((int)bits, l);
        int skip = v - (__builtin_amdgcn_readlane(upto, l) - __popc(word));
        for (; skip > 0; --skip) word &= word - 1;
        return nct + 32 * (base + l) + __builtin_ctz(word);
      }
      v -= __builtin_amdgcn_readlane(upto, 63);
    }
    return nct + this->nht;
  }
  // The first tile from t on that is not skipped (its class in cls), or t_end.
  __device__ __forceinline__ int find_tile(int t, int &cls) {
    while (t < t_end) {
      if (t >= wbase + 64) window(t);
      const uint64_t m = wseen >> (t - wbase);
      if (m) {
        t += __builtin_ctzll(m);
        cls = (wmixed >> (t - wbase)) & 1 ? TILE_MIXED : TILE_FULL;
        return t;
      }
      t = wbase + 64;
      if constexpr (MK == PF_ARITH) {
        // The causal rule hides every tile after the first hidden one.
        if (this->causal && t >= nct && (t - nct) * kPfKeys > this->qlast + this->off) return t_end;
      }
    }
    return t_end;
  }
  static __device__ __forceinline__ int xv(int r) { return CP == 16 ? r & 3 : CP == 8 ? (r >> 1) & 1 : 0; }

  // Starts tile t's loads into LDS (rows past the segment's end repeat its
  // last row; their scores get a -inf bias, as such a tile is MIXED).
  __device__ __forceinline__ void load_tile(int t, uint16_t *ks, uint16_t *vs) const {
    const bool cold = t < nct;
    const int key0 = (cold ? t : t - nct) * kPfKeys, last = (cold ? p.cold_len : p.hot_len) - key0 - 1;
    const uint32_t krs = cold ? D * 2 : (uint32_t)p.hks2 * 2, vrs = cold ? D * 2 : (uint32_t)p.hvs2 * 2;
    const auto rk = tile_rsrc((cold ? cold_kb : hot_kb) + (int64_t)key0 * krs, 0xffffffffu);
    const auto rv = tile_rsrc((cold ? cold_vb : hot_vb) + (int64_t)key0 * vrs, 0xffffffffu);
    auto load = [&](__amdgpu_buffer_rsrc_t rs, uint16_t *to, int j, uint32_t voff, uint32_t soff) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t *)(to + (j * 4 + wave) * 512), 16, (int)voff, (int)soff,
                                               0, 0);
    };
    if (last >= kPfKeys - 1) {
      // A whole tile: one lane offset each, the instructions' rows in the
      // scalar offset.
      const uint32_t ko = (uint32_t)lrow * krs + (uint32_t)kc, vo = (uint32_t)lrow * vrs + (uint32_t)vc;
#pragma unroll
      for (int j = 0; j < NJ; ++j) load(rk, ks, j, ko, (uint32_t)(j * 4 * RPI) * krs);
#pragma unroll
      for (int j = 0; j < NJ; ++j) load(rv, vs, j, vo, (uint32_t)(j * 4 * RPI) * vrs);
      return;
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) load(rk, ks, j, (uint32_t)min(lrow + j * 4 * RPI, last) * krs + (uint32_t)kc, 0);
#pragma unroll
    for (int j = 0; j < NJ; ++j) load(rv, vs, j, (uint32_t)min(lrow + j * 4 * RPI, last) * vrs + (uint32_t)vc, 0);
  }

  __device__ __forceinline__ void load_q(uint4 (&qx)[KS]) const {
    const char *qrow = p.q + ((int64_t)b * p.qs0 + (int64_t)h * p.qs1 + (int64_t)qc * p.qs2) * 2 + 16 * hf;
#pragma unroll
    for (int st = 0; st < KS; ++st) qx[st] = load16(qrow + 32 * st);
  }

  // Visible keys of MIXED tile t as bits, 64 a query row of the block, into
  // vis[ROWS][2] (thread tid: row tid / 2, keys 32 (tid % 2) .. + 31).  Read
  // by every lane of the row in hide(); the registers of the mask's elements
  // are then not live beside the tile's operands.
  __device__ __forceinline__ void visible_bits(int t, uint32_t *vis) const {
    const bool cold = t < nct;
    const int key0 = (cold ? t : t - nct) * kPfKeys, n = (cold ? p.cold_len : p.hot_len) - key0;
    const int tid = this->tid, half = tid & 1, qr = min(q0 + (tid >> 1), p.qlen - 1);
    int seen = n;  // keys [0, seen) of the tile can be visible
    if (!cold && this->causal) seen = min(seen, qr + this->off - key0 + 1);
    const int cnt = min(max(seen - 32 * half, 0), 32);
    uint32_t bits = cnt == 32 ? ~0u : (1u << cnt) - 1u;
    if (MK == PF_BOOL && !cold && cnt > 0) {
      const char *m = p.mask + mask_off(p, b, h, qr, key0 + 32 * half);
      uint32_t on = 0;
      if (p.ms3 == 1 && cnt == 32) {
        const uint4 lo = load_any<uint4>(m), hi = load_any<uint4>(m + 16);
        const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) on |= (w[u] >> (8 * i)) & 0xffu ? 1u << (4 * u + i) : 0u;
      } else {
        for (int i = 0; i < cnt; ++i) on |= m[(int64_t)i * p.ms3] ? 1u << i : 0u;
      }
      bits &= on;
    }
    vis[tid] = bits;
  }
  // Hidden keys' dot products become -inf; the others stay as in a FULL
  // tile, bit for bit.
  __device__ __forceinline__ void hide(f32x16_t (&s)[2], const uint32_t *vis) const {
    const uint2 w = *reinterpret_cast<const uint2 *>(vis + 2 * (32 * wave + row));
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const uint32_t v = (sub ? w.y : w.x) >> (4 * hf);  // bit 8 u + i: key 8 u + 4 hf + i
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (!(v & (1u << (8 * (i >> 2) + (i & 3))))) s[sub][i] = -INFINITY;
    }
  }
  // MIXED tile t under a float mask: scores become s * scaling * log2 e +
  // bias (base 2).
  __device__ __forceinline__ void add_bias(f32x16_t (&s)[2], int t) const {
    const bool cold = t < nct;
    const int key0 = (cold ? t : t - nct) * kPfKeys, n = (cold ? p.cold_len : p.hot_len) - key0;
    const int64_t row_mo = this->row_mask_off(qc);
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float bias[4];
        this->bias4(cold, key0, n, 32 * sub + 8 * u + 4 * hf, qc, row_mo, bias);
#pragma unroll
        for (int i = 0; i < 4; ++i) s[sub][4 * u + i] = fmaf(s[sub][4 * u + i], p.scale_log2, bias[i]);
      }
  }

  // The rows' outputs (dims 32 dt + 8 u + 4 hf .. + 3 of the lane's row), or
  // (partial >= 0) the unnormalised sums, running max and row sum.
  __device__ __forceinline__ void finish(const f32x16_t (&o)[ND], float m_run, float l_lane, int partial) const {
    const float l_row = half_wave_sum(l_lane);
    if (qi >= p.qlen) return;
    if (partial >= 0) {
      const int64_t sr = (int64_t)partial * p.part_rows + 32 * wave + row;
      float *po = p.ws_o + sr * D;
#pragma unroll
      for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          *reinterpret_cast<f32x4_t *>(po + 32 * dt + 8 * u + 4 * hf) =
              f32x4_t{o[dt][4 * u], o[dt][4 * u + 1], o[dt][4 * u + 2], o[dt][4 * u + 3]};
      if (hf == 0) {
        p.ws_m[sr] = m_run;
        p.ws_l[sr] = l_row;
      }
      return;
    }
    // A row with no visible key (fully masked) gets zeros.
    const float inv = l_row > 0.f ? 1.f / l_row : 0.f;
    char *orow = this->out_row(qi);
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        *reinterpret_cast<uint2 *>(orow + (32 * dt + 8 * u + 4 * hf) * 2) =
            make_uint2(pack2<DT>(o[dt][4 * u] * inv, o[dt][4 * u + 1] * inv),
                       pack2<DT>(o[dt][4 * u + 2] * inv, o[dt][4 * u + 3] * inv));
  }

  // One tile, its rows in ks / vs.
  __device__ __forceinline__ void tile(int t, int cls, const uint16_t *ks, const uint16_t *vs, const uint32_t *vis,
                                       const uint4 (&qx)[KS], f32x16_t (&o)[ND], float &m_run, float &l_lane) const {
    const char *kb = reinterpret_cast<const char *>(ks), *vb = reinterpret_cast<const char *>(vs);
    f32x16_t s[2] = {};
    // Operand i (step i / 2, sub-tile i % 2): kAhead reads in flight, one more
    // issued behind each matrix instruction, in that order.
    constexpr int NR = 2 * KS, kAhead = NR < 6 ? NR : 6;
    auto k_op = [&](int i) {
      return *reinterpret_cast<const uint4 *>(kb + (kaddr ^ ((i >> 1) << 5)) + (i & 1) * 32 * CP * 16);
    };
    uint4 ka[NR];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) ka[i] = k_op(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      s[i & 1] = mfma_32x32x16<DT>(ka[i], qx[i >> 1], s[i & 1]);
      if (i + kAhead < NR) ka[i + kAhead] = k_op(i + kAhead);
      __builtin_amdgcn_sched_barrier(0);
    }
    // The first PV step's V operands, in flight under the softmax.
    uint4 va[2][ND];
    load_v(vb, 0, va[0]);
    __builtin_amdgcn_sched_barrier(0);
    // Scores in base-2 units are cc * s, cc = scaling * log2 e folded into
    // the exponent (1 where a float mask's bias was added).
    float cc = p.scale_log2;
    if (cls == TILE_MIXED) {
      if constexpr (MK == PF_FLOAT) {
        add_bias(s, t);
        cc = 1.f;
      } else {
        hide(s, vis);
      }
    }
    // The running max is raised (and the sums rescaled) only on a tile where
    // a lane's maximum exceeds it by more than 2^kRescaleSlack; the row's
    // maximum, over its two lanes, is formed on such tiles alone.
    float x = s[0][0];
#pragma unroll
    for (int i = 1; i < 16; ++i) x = fmaxf(x, s[0][i]);
#pragma unroll
    for (int i = 0; i < 16; ++i) x = fmaxf(x, s[1][i]);
    if (__ballot(x * cc > m_run + kRescaleSlack)) {
      const float mt = half_wave_max(x) * cc;
      const float m_new = mt > m_run + kRescaleSlack ? mt : m_run;
      const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_lane *= alpha;
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) o[dt] *= alpha;
      m_run = m_new;
    }
    // Probabilities 2^(cc s - m), rounded to the dtype as operands; a row
    // that has seen no key keeps m = -inf, its probabilities are 0.
    // Four steps of 16 keys: a step's matrix instructions issue among the
    // next step's exponentials, and its V operands were read a step before.
    const float m_neg = m_run == -INFINITY ? 0.f : -m_run;
    auto probs = [&](int k) {
      float e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) e[i] = __builtin_amdgcn_exp2f(fmaf(s[k >> 1][8 * (k & 1) + i], cc, m_neg));
#pragma unroll
      for (int i = 0; i < 8; ++i) l_lane += e[i];
      return make_uint4(pack2<DT>(e[0], e[1]), pack2<DT>(e[2], e[3]), pack2<DT>(e[4], e[5]), pack2<DT>(e[6], e[7]));
    };
    uint4 pb = probs(0);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      __builtin_amdgcn_sched_barrier(0);
      if (k < 3) load_v(vb, k + 1, va[(k + 1) & 1]);
      uint4 pn = pb;
      if (k < 3) pn = probs(k + 1);
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) o[dt] = mfma_32x32x16<DT>(va[k & 1][dt], pb, o[dt]);
      if (k < 3) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * ND, 0);
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x402, 28 / ND, 0);
        }
      }
      pb = pn;
    }
  }
  // V^T operands of PV step k (keys 16 k .. + 15 of the tile).
  __device__ __forceinline__ void load_v(const char *vb, int k, uint4 (&a)[ND]) const {
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) {
      const char *at = vb + vaddr[dt] + 16 * k * CP * 16;
      const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t *)at));
      const uint2 hi =
          __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t *)(at + 8 * CP * 16)));
      a[dt] = make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
  }
};

// Blocks are dealt to the eight dies in turn: a die takes consecutive
// shares, which read the same heads' keys through its L2.
__device__ __forceinline__ int die_order(int blocks) {
  const int i = (int)blockIdx.x;
  return blocks > 0 && !(blocks & 7) ? (i & 7) * (blocks >> 3) + (i >> 3) : i;
}

// Mask tensors: the weights of the units from the bits of their visible
// tiles, kept as prefix sums over the mask's own (batch, head) planes: pre[u]
// before row block u % nrb of plane u / nrb.  The heads that share a plane
// repeat it.  A unit that sees no tile weighs one, so that a block writes its
// rows.  (Shares by the causal rule's weights whatever the mask, where the
// block that reached a unit's end took all the tiles past the diagonal: 4096
// positions of 12 heads over 8192 keys, all visible 291 us a call, 240 by the
// table; columns from the diagonal on 181 -> 110; documents of 512 tokens 61
// -> 43.  The table costs a block about 3 us, mostly its code's first run, and
// the test for the causal tiles about 1.)
struct PfTable {
  const PrefillParams &p;
  const int *pre;
  const int own, rep;  // own row blocks; heads that repeat a plane
  __device__ __forceinline__ int at(int i) const { return __builtin_amdgcn_readfirstlane(pre[i]); }
  __device__ __forceinline__ int first_own(int b, int h) const {
    return ((p.mask_b == 1 ? 0 : b) * p.mask_h + (p.mask_h == 1 ? 0 : h)) * p.sh.nrb;
  }
  // Weights before batch row b.
  __device__ __forceinline__ int batch_start(int b) const {
    return p.mask_b == 1 ? b * rep * at(own) : rep * at(b * p.mask_h * p.sh.nrb);
  }
  __device__ __forceinline__ int total() const { return (p.mask_b == 1 ? p.batch : 1) * rep * at(own); }
  // Weights [us, ue) of unit (bh, rb).
  __device__ __forceinline__ void unit(int bh, int rb, int &us, int &ue) const {
    const int b = bh / p.hq, h = bh - b * p.hq, o = first_own(b, h);
    const int before = p.mask_h == 1 ? h * (at(o + p.sh.nrb) - at(o)) - at(o)
                                     : -at(p.mask_b == 1 ? 0 : b * p.mask_h * p.sh.nrb);
    us = batch_start(b) + before + at(o + rb);
    ue = batch_start(b) + before + at(o + rb + 1);
  }
  // Of own row blocks [o, o + n): the last that starts at or before x.
  __device__ __forceinline__ int find(int o, int n, int x) const {
    const int lane = threadIdx.x & 63;
    int i = 0;
    for (int base = 0; base < n; base += 64) {
      const uint64_t m = __ballot(base + lane < n && pre[o + min(base + lane, n - 1)] <= x);
      i += __popcll(m);
      if (m != ~uint64_t(0)) break;
    }
    return o + i - 1;
  }
  // The unit that weight w < total() falls in.
  __device__ __forceinline__ void unit_of(int w, int &bh, int &rb) const {
    const int nrb = p.sh.nrb;
    int b = 0;
    if (p.mask_b == 1) {
      b = w / (rep * at(own));
    } else {
      while (b + 1 < p.batch && batch_start(b + 1) <= w) ++b;
    }
    const int o = first_own(b, 0);
    int r = w - batch_start(b);
    if (p.mask_h == 1) {
      const int plane = at(o + nrb) - at(o), h = r / plane;
      rb = find(o, nrb, at(o) + r - h * plane) - o;
      bh = b * p.hq + h;
    } else {
      const int u = find(o, p.hq * nrb, at(o) + r) - o, h = u / nrb;
      rb = u - h * nrb;
      bh = b * p.hq + h;
    }
  }
};

// Word i of a mask tensor's own row blocks' bits, both 64-row entries.
__device__ __forceinline__ uint32_t own_bits(const PrefillParams &p, int i) {
  const int words = 1 << p.seen_shift;
  const uint32_t *row = p.seen + ((int64_t)(i >> p.seen_shift) << (p.seen_shift + 1)) + (i & (words - 1));
  return row[0] | row[words];
}
// Whether every row block of a mask tensor sees just the tiles that the causal
// rule's weights count (p.sh): the shares need no table then.  Called by the
// whole block; bits: own_bits of the thread's first word.
__device__ __forceinline__ bool sees_causal_tiles(const PrefillParams &p, int own, uint32_t bits) {
  __shared__ int other[kPfThreads / 64];
  const int nct = (p.cold_len + kPfKeys - 1) / kPfKeys, nrb = p.sh.nrb;
  bool differs = false;
  for (int i = threadIdx.x; i < own << p.seen_shift; i += kPfThreads) {
    if (i >= kPfThreads) bits = own_bits(p, i);
    const int u = i >> p.seen_shift, at = i & ((1 << p.seen_shift) - 1);
    const int n = p.sh.weight(own == nrb ? u : u % nrb) - nct - 32 * at;  // tiles from the word's first on
    differs |= bits != (n >= 32 ? ~0u : n <= 0 ? 0u : (1u << n) - 1u);
  }
  const uint64_t any = __ballot(differs);
  if ((threadIdx.x & 63) == 0) other[threadIdx.x >> 6] = any != 0;
  __syncthreads();
  int all = 0;
#pragma unroll
  for (int i = 0; i < kPfThreads / 64; ++i) all |= other[i];
  return __builtin_amdgcn_readfirstlane(all) == 0;
}

// Fills pre[0 .. own] by the whole block.
__device__ __forceinline__ void fill_table(const PrefillParams &p, int *pre, int own) {
  __shared__ int wsum[kPfThreads / 64];
  const int tid = threadIdx.x, wave = tid >> 6;
  const int nct = (p.cold_len + kPfKeys - 1) / kPfKeys;
  // 1 << ls lanes a unit, a word of its two rows each at a time.
  const int ls = min(p.seen_shift, 6), sub = tid & ((1 << ls) - 1);
  for (int u = tid >> ls; u < own; u += kPfThreads >> ls) {
    const uint32_t *row = p.seen + ((int64_t)u << (p.seen_shift + 1));
    int n = 0;
    for (int i = sub; i < 1 << p.seen_shift; i += 64) n += __popc(row[i] | row[i + (1 << p.seen_shift)]);
    for (int o = 1; o < 1 << ls; o <<= 1) n += __shfl_xor(n, o, 64);
    if (sub == 0) pre[u] = max(1, nct + n);
  }
  __syncthreads();
  constexpr int PT = kPfMaxUnits / kPfThreads;  // row blocks a thread
  int x[PT], mine = 0;
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    x[j] = PT * tid + j < own ? pre[PT * tid + j] : 0;
    mine += x[j];
  }
  const int upto = wave_incl_scan(mine);
  if ((tid & 63) == 63) wsum[wave] = upto;
  __syncthreads();
  int at = upto - mine;
#pragma unroll
  for (int i = 0; i < kPfThreads / 64 - 1; ++i) at += i < wave ? wsum[i] : 0;
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    if (PT * tid + j <= own) pre[PT * tid + j] = at;
    at += x[j];
  }
  __syncthreads();
}

template <int DT, int KT, int MK>
__global__ void __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(2)))
prefill_attn32_kernel(PrefillParams p) {
  using Blk = PfBlock32<DT, KT, MK>;
  // Two buffers as objects of their own: the compiler then knows that a
  // tile's operand reads do not depend on the other buffer's loads.
  __shared__ __align__(1024) uint16_t k0[Blk::TILE], k1[Blk::TILE], v0[Blk::TILE], v1[Blk::TILE];
  __shared__ uint32_t vis0[2 * Blk::ROWS], vis1[2 * Blk::ROWS];
  // Mask tensors: the units' weights (else arithmetic, see PfShares).
  constexpr bool kTable = MK != PF_ARITH;
  __shared__ int pre[kTable ? kPfMaxUnits : 1];
  const PfTable tab{p, pre, p.mask_b * p.mask_h * p.sh.nrb, p.mask_h == 1 ? p.hq : 1};
  uint32_t bits = 0u;
  if (kTable && p.sh.blocks > 0 && (int)threadIdx.x < tab.own << p.seen_shift) bits = own_bits(p, threadIdx.x);
  // This block's units: a share's range of weights [w, w_end), or one unit.
  int bh, rb, w, w_end, id = die_order(p.sh.blocks);
  p.sh.first(id, p.batch * p.hq, bh, rb, w, w_end);
  Blk blk(p);
  bool table = false;
  if constexpr (kTable) table = p.sh.blocks > 0 && !sees_causal_tiles(p, tab.own, bits);
  if (table) {
    PfShares sh = p.sh;
    fill_table(p, pre, tab.own);
    const int total = tab.total(), units = p.batch * p.hq * sh.nrb;
    sh.deal(total, (int)pf_min(sh.blocks, share_blocks_of(total, units, sh.slots)));
    if ((int)blockIdx.x >= sh.blocks) return;
    id = die_order(sh.blocks);
    w = sh.start(id);
    w_end = sh.start(id + 1);
    tab.unit_of(w, bh, rb);
  }
  const int w0 = w;
  while (w < w_end) {
    int us, ue;
    if (table) {
      tab.unit(bh, rb, us, ue);
    } else {
      us = p.sh.unit_start(bh, rb);
      ue = us + p.sh.weight(rb);
    }
    const bool ends = w_end >= ue;
    const int frag = 2 * id + (w == w0 ? 0 : 1), partial = w == us && ends ? -1 : frag;
    if (p.cuts && threadIdx.x == 0) {
      int2 &cut = p.cuts[bh * p.sh.nrb + rb];
      if (w == us) cut.x = frag;
      if (ends) cut.y = id;
    }
    // Under a table a fragment is the unit's visible tiles [w - us, w_end - us);
    // else all are visible up to there.
    blk.set_unit(bh, rb, w - us, ends ? p.sh.tiles : w_end - us);
    if (table) {
      bits = blk.seen_bits(0);
      if (w > us) blk.t_begin = blk.locate(w - us, bits);
      if (!ends) blk.t_end = blk.locate(w_end - us, bits);
    }
    blk.window(blk.t_begin);
    int cls = TILE_FULL, t = blk.find_tile(blk.t_begin, cls);
    if (t < blk.t_end) blk.load_tile(t, k0, v0);
    uint4 qx[Blk::KS];
    blk.load_q(qx);
    f32x16_t o[Blk::ND] = {};
    float m_run = -INFINITY, l_lane = 0.f;  // l_lane: this lane's share of the row sum
    // The tile's loads have arrived (each wave waits for its own, then the
    // barrier), and every wave is done with the buffer the next ones fill:
    // its reads of the tile before are issued ahead of the wait, which no
    // memory access is moved across, and the wait covers them too.
    auto step = [&](uint16_t *ks, uint16_t *vs, uint16_t *kn, uint16_t *vn, uint32_t *vis) {
      int cls_n = TILE_FULL;
      const int tn = blk.find_tile(t + 1, cls_n);
      if (MK != PF_FLOAT && cls == TILE_MIXED) blk.visible_bits(t, vis);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(kWaitMem);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (tn < blk.t_end) blk.load_tile(tn, kn, vn);
      blk.tile(t, cls, ks, vs, vis, qx, o, m_run, l_lane);
      t = tn;
      cls = cls_n;
    };
    while (t < blk.t_end) {
      step(k0, v0, k1, v1, vis0);
      if (t >= blk.t_end) break;
      step(k1, v1, k0, v0, vis1);
    }
    blk.finish(o, m_run, l_lane, partial);
    w = ue;
    if (++rb == p.sh.nrb) {
      rb = 0;
      ++bh;
    }
    if (w < w_end) __syncthreads();  // the next unit's first loads reuse the LDS
  }
}

// Merges the units that the shares cut: out = sum_i 2^(m_i - M) o_i / sum_i
// 2^(m_i - M) l_i over a unit's partials, M their largest running max.
// Grid (pieces of rows, units): D / 4 threads per output row, 4 dims each;
// blocks of whole units leave at once.  A row that saw no key gets zeros.
constexpr int kMergeBatch = 4;
template <int DT>
__global__ void __launch_bounds__(kPfThreads) prefill_merge_kernel(PrefillParams p, int D) {
  const int nrb = p.sh.nrb, bh = blockIdx.y / nrb, rb = blockIdx.y - bh * nrb;
  const int2 cut = p.cuts[blockIdx.y];
  const int i0 = cut.x >> 1, i1 = cut.y;
  if (i0 == i1) return;
  const int tpr = D / 4, rows_per_block = kPfThreads / tpr;
  const int r = blockIdx.x * rows_per_block + threadIdx.x / tpr, d0 = 4 * (threadIdx.x % tpr);
  const int qi = rb * kPfUnitRows + r;
  if ((int)threadIdx.x >= rows_per_block * tpr || r >= kPfUnitRows || qi >= p.qlen) return;
  auto at = [&](int i) { return (int64_t)(i == i0 ? cut.x : 2 * i) * p.part_rows + r; };
  // kMergeBatch partials' loads in flight together, folded by their largest
  // max (a unit of 9 partials, 28 x 16 rows: 10.6 us reading one at a time,
  // 4.0 in batches).
  float M = -INFINITY, L = 0.f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int f = i0; f <= i1; f += kMergeBatch) {
    float ms[kMergeBatch], ls[kMergeBatch];
    f32x4_t os[kMergeBatch];
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const bool in = f + u <= i1;
      const int64_t x = at(in ? f + u : f);
      ms[u] = in ? p.ws_m[x] : -INFINITY;
      ls[u] = in ? p.ws_l[x] : 0.f;
      os[u] = in ? *reinterpret_cast<const f32x4_t *>(p.ws_o + x * D + d0) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    float m = M;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) m = fmaxf(m, ms[u]);
    if (m == -INFINITY) continue;
    const float w0 = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M - m);
    L *= w0;
    acc *= w0;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const float w = ms[u] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms[u] - m);
      L = fmaf(w, ls[u], L);
      acc += w * os[u];
    }
    M = m;
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  const int b = bh / p.hq, h = bh - b * p.hq;
  *reinterpret_cast<uint2 *>(p.out + ((((int64_t)b * p.qlen + qi) * p.hq + h) * D + d0) * 2) =
      make_uint2(pack2<DT>(acc[0] * inv, acc[1] * inv), pack2<DT>(acc[2] * inv, acc[3] * inv));
}

// Head dims above 128, one tile at a time, every step in order: store the
// tile to LDS, scores, softmax, PV.
template <int DT, int KT, int MK>
__global__ void __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(2)))
prefill_attn_kernel(PrefillParams p) {
  using Blk = PfBlock<DT, KT, MK>;
  constexpr int D = Blk::D;
  __shared__ __align__(16) uint16_t ks[Blk::KTILE];
  __shared__ __align__(16) uint16_t vt[Blk::VTILE];
  __shared__ uint8_t tcls[MK == PF_ARITH ? 1 : kPfLdsTiles];
  Blk blk(p, tcls);
  uint4 qx[KT];
  blk.load_q(qx);
  f32x4_t o[D / 16];
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) o[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_lane = 0.f;  // l_lane: this lane's share of the row sum
  int t = blk.first_tile();
  if (t < blk.t_end) {
    blk.load_k(t);
    blk.load_v(t);
  }
  while (t < blk.t_end) {
    const int cls = blk.tile_class(t), tn = blk.next_tile(t);
    __syncthreads();  // the previous tile's reads of ks / vt are done
    blk.store_k(ks);
    blk.store_v(vt);
    __syncthreads();
    if (tn < blk.t_end) {
      blk.load_k(tn);
      blk.load_v(tn);
    }
    // Scores in base-2 units are cc * s: FULL tiles keep the raw dot products
    // (cc = scaling * log2 e, folded into the exponent), MIXED tiles add the
    // bias first (cc = 1).
    f32x4_t s[4];
    pf_scores<DT, KT>(s, ks, qx, blk.col, blk.grp);
    float cc = p.scale_log2;
    if (cls == TILE_MIXED) {
      blk.add_bias(s, t);
      cc = 1.f;
    }
    pf_max_raise<D / 16>(s, cc, m_run, l_lane, o);
    uint4 pb[2];
    pf_probs<DT>(s, cc, m_run, l_lane, pb);
    pf_pv<DT, D>(o, pb, vt, blk.col, blk.grp);
    t = tn;
  }
  blk.finish(o, m_run, l_lane);
}

// Head dims above 128: merges the key splits, out = sum_s 2^(m_s - M) o_s / sum_s 2^(m_s - M) l_s
// with M the largest running max.  D / 4 threads per output row, 4 dims
// each; a row that saw no key in any split gets zeros.
template <int DT>
__global__ void __launch_bounds__(kPfThreads) prefill_combine_kernel(PrefillParams p, int D) {
  const int tpr = D / 4, rows_per_block = kPfThreads / tpr;
  if ((int)threadIdx.x >= rows_per_block * tpr) return;
  const int64_t nrows = (int64_t)p.batch * p.qlen * p.hq;
  const int64_t row = (int64_t)blockIdx.x * rows_per_block + threadIdx.x / tpr;
  const int d0 = 4 * (threadIdx.x % tpr);
  if (row >= nrows) return;
  float M = -INFINITY;
  for (int sp = 0; sp < p.nsplit; ++sp) M = fmaxf(M, p.ws_m[sp * nrows + row]);
  float L = 0.f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  if (M != -INFINITY) {
    for (int sp = 0; sp < p.nsplit; ++sp) {
      const float m = p.ws_m[sp * nrows + row];
      if (m == -INFINITY) continue;
      const float w = __builtin_amdgcn_exp2f(m - M);
      L += w * p.ws_l[sp * nrows + row];
      acc += w * *reinterpret_cast<const f32x4_t *>(p.ws_o + (sp * nrows + row) * D + d0);
    }
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  *reinterpret_cast<uint2 *>(p.out + (row * D + d0) * 2) =
      make_uint2(pack2<DT>(acc[0] * inv, acc[1] * inv), pack2<DT>(acc[2] * inv, acc[3] * inv));
}

static int64_t div_up(int64_t a, int64_t b) { return pf_div_up(a, b); }

// Key splits of head dims above 128: enough (row block, batch row * head,
// split) units for about two rounds of the GPU's block slots, at least two
// key tiles per split, at most 8.  With the longest-first order a second
// round fills the slots the short row blocks free; more splits only add
// partial rows to write and merge.
static int prefill_splits(int Q, int rows, int BH, int cold_len, int hot_len, int slots) {
  const int64_t units = div_up(Q, rows) * BH, tiles = div_up(cold_len, kPfKeys) + div_up(hot_len, kPfKeys);
  if (units >= 2 * (int64_t)slots) return 1;
  const int64_t want = div_up(2 * (int64_t)slots, units), most = std::max<int64_t>(1, tiles / 2);
  return (int)std::max<int64_t>(1, std::min<int64_t>({want, most, 8}));
}

// Block slots of the attention kernel: two blocks per compute unit.
static int prefill_slots() { return 2 * device_cu_count(); }

// Rows of a partial: a unit's, of which one row block alone has only Q.
static int part_rows(int Q) { return std::min(Q, kPfUnitRows); }

struct PrefillWorkspace {
  size_t tiles_bytes, seen_off, cuts_off, m_off, l_off, o_off, total;
  int nsplit, blocks, seen_shift;
};

static PrefillWorkspace prefill_workspace(int B, int hq, int D, int Q, int cold_len, int hot_len, int mask_b,
                                          int mask_h) {
  PrefillWorkspace w;
  const bool shares = D <= 128;
  w.nsplit = shares ? 1 : prefill_splits(Q, 64, B * hq, cold_len, hot_len, prefill_slots());
  w.blocks = shares ? prefill_share_blocks(Q, B * hq, cold_len, hot_len, prefill_slots()) : 0;
  w.tiles_bytes = hot_len > 0 ? (size_t)mask_b * mask_h * div_up(Q, kPfRows) * div_up(hot_len, kPfKeys) : 0;
  // Partial rows: every row of each split, or two units a share.
  const size_t nrows = shares ? (size_t)2 * w.blocks * part_rows(Q) : w.nsplit > 1 ? (size_t)B * Q * hq * w.nsplit : 0;
  // With shares: the bits of a mask tensor's visible tiles and the units' cuts.
  const int64_t nrb = div_up(Q, kPfUnitRows), words = div_up(div_up(hot_len, kPfKeys), 32);
  for (w.seen_shift = 0; (int64_t(1) << w.seen_shift) < words;) ++w.seen_shift;
  const size_t seen = w.blocks > 0 && w.tiles_bytes > 0 ? ((size_t)mask_b * mask_h * nrb * 8) << w.seen_shift : 0;
  const size_t cuts = w.blocks > 0 ? (size_t)B * hq * nrb * sizeof(int2) : 0;
  w.seen_off = (w.tiles_bytes + 255) & ~size_t(255);
  w.cuts_off = w.seen_off + ((seen + 255) & ~size_t(255));
  w.m_off = w.cuts_off + ((cuts + 255) & ~size_t(255));
  w.l_off = w.m_off + ((nrows * 4 + 255) & ~size_t(255));
  w.o_off = w.l_off + ((nrows * 4 + 255) & ~size_t(255));
  w.total = nrows > 0 ? w.o_off + nrows * D * 4 : w.tiles_bytes;
  return w;
}

}  // namespace kiv

using namespace kiv;

extern "C" {

size_t kiv_prefill_workspace_size(int32_t batch, int32_t num_q_heads, int32_t head_dim, int32_t q_len,
                                  int32_t cold_len, int32_t hot_len) {
  if (batch < 1 || num_q_heads < 1 || head_dim < 1 || q_len < 1 || cold_len < 0 || hot_len < 0) return 0;
  return prefill_workspace(batch, num_q_heads, head_dim, q_len, cold_len, hot_len, batch, num_q_heads).total;
}

int kiv_prefill_attention(const kiv_attention_args_t *a, kiv_stream_t stream) {
  const char *who = "kiv_prefill_attention";
  if (!a) return fail(KIV_ERR_INVALID, "%s: null argument", who);
  const int dt = a->dtype;
  if (dt != KIV_DTYPE_F16 && dt != KIV_DTYPE_BF16) return fail(KIV_ERR_UNSUPPORTED, "%s: fp16/bf16 only", who);
  const int B = a->batch, hq = a->num_q_heads, hkv = a->num_kv_heads, D = a->head_dim, Q = a->q_len;
  if (B < 1 || hq < 1 || hkv < 1 || Q < 1 || hq % hkv) return fail(KIV_ERR_INVALID, "%s: bad head geometry", who);
  const int kt = D / 32;
  if (D % 32 || !(kt <= 4 || kt == 6 || kt == 8))
    return fail(KIV_ERR_UNSUPPORTED, "%s: head_dim %d unsupported (32, 64, 96, 128, 192, 256)", who, D);
  if (a->cold_len < 0 || a->hot_len < 0 || a->cold_len + a->hot_len < 1)
    return fail(KIV_ERR_INVALID, "%s: no keys", who);
  const bool need_cold = a->cold_len > 0, need_hot = a->hot_len > 0;
  if (!a->q || !a->out || (need_cold && (!a->cold_k || !a->cold_v)) || (need_hot && (!a->hot_k || !a->hot_v)))
    return fail(KIV_ERR_INVALID, "%s: null pointer", who);
  if (a->q_stride[3] != 1) return fail(KIV_ERR_INVALID, "%s: q head_dim stride must be 1", who);
  const uintptr_t ptrs = (uintptr_t)a->q | (uintptr_t)a->out |
                         (need_cold ? (uintptr_t)a->cold_k | (uintptr_t)a->cold_v : 0) |
                         (need_hot ? (uintptr_t)a->hot_k | (uintptr_t)a->hot_v : 0);
  if (ptrs & 15) return fail(KIV_ERR_INVALID, "%s: q, K, V and out must be 16-byte aligned", who);
  for (int i = 0; i < 3; ++i)
    if ((a->q_stride[i] % 8) || (a->hot_k_stride[i] % 8) || (a->hot_v_stride[i] % 8))
      return fail(KIV_ERR_INVALID, "%s: strides must be multiples of 8 elements", who);
  if ((int64_t)B * hq > 65535) return fail(KIV_ERR_UNSUPPORTED, "%s: batch * heads above 65535", who);
  // Row offsets within a tile are 32-bit; the softmax takes the row maximum
  // of the unscaled dot products, which needs a positive scale.
  if (a->hot_k_stride[2] >= (1 << 24) || a->hot_v_stride[2] >= (1 << 24))
    return fail(KIV_ERR_UNSUPPORTED, "%s: hot row stride too large", who);
  if (!(a->scaling > 0.f)) return fail(KIV_ERR_UNSUPPORTED, "%s: scaling must be positive", who);
  int mk = a->mask_kind;
  const bool explicit_mask = a->mask != nullptr;
  if (explicit_mask) {
    if (mk < KIV_MASK_BOOL || mk > KIV_MASK_BF16) return fail(KIV_ERR_INVALID, "%s: unknown mask kind %d", who, mk);
    if (!need_hot) mk = KIV_MASK_NONE;  // the mask covers hot columns only
  } else if (mk != KIV_MASK_CAUSAL) {
    mk = KIV_MASK_NONE;
  }
  PrefillParams p;
  p.q = (const char *)a->q;
  p.qs0 = a->q_stride[0];
  p.qs1 = a->q_stride[1];
  p.qs2 = a->q_stride[2];
  p.cold_k = (const char *)a->cold_k;
  p.cold_v = (const char *)a->cold_v;
  p.cold_len = a->cold_len;
  p.hot_len = a->hot_len;
  p.hot_k = (const char *)a->hot_k;
  p.hot_v = (const char *)a->hot_v;
  p.hks0 = a->hot_k_stride[0];
  p.hks1 = a->hot_k_stride[1];
  p.hks2 = a->hot_k_stride[2];
  p.hvs0 = a->hot_v_stride[0];
  p.hvs1 = a->hot_v_stride[1];
  p.hvs2 = a->hot_v_stride[2];
  p.mask = (const char *)a->mask;
  p.mask_kind = mk;
  p.ms0 = a->mask_stride[0];
  p.ms1 = a->mask_stride[1];
  p.ms2 = a->mask_stride[2];
  p.ms3 = a->mask_stride[3];
  p.mask_vec4 = mk == KIV_MASK_BOOL && p.ms3 == 1 && !(((uintptr_t)a->mask | p.ms0 | p.ms1 | p.ms2) & 3);
  p.mask_b = p.ms0 == 0 ? 1 : B;
  p.mask_h = p.ms1 == 0 ? 1 : hq;
  p.tiles = nullptr;
  p.batch = B;
  p.hq = hq;
  p.hkv = hkv;
  p.qlen = Q;
  p.scale_log2 = a->scaling * kLog2e;
  p.out = (char *)a->out;
  hipStream_t st = (hipStream_t)stream;
  const int mode = mk == KIV_MASK_BOOL ? PF_BOOL : (mk == KIV_MASK_NONE || mk == KIV_MASK_CAUSAL) ? PF_ARITH : PF_FLOAT;
  const PrefillWorkspace w = prefill_workspace(B, hq, D, Q, a->cold_len, a->hot_len,
                                               mode != PF_ARITH ? p.mask_b : 0, mode != PF_ARITH ? p.mask_h : 0);
  p.nsplit = w.nsplit;
  p.sh = prefill_shares(Q, B * hq, a->cold_len, a->hot_len, mk != KIV_MASK_NONE, w.blocks, prefill_slots());
  p.part_rows = part_rows(Q);
  p.ws_m = p.ws_l = p.ws_o = nullptr;
  if (w.total > 0 && (!a->workspace || a->workspace_bytes < w.total || ((uintptr_t)a->workspace & 255)))
    return fail(KIV_ERR_INVALID, "%s: needs a 256-byte aligned workspace of %zu bytes (kiv_prefill_workspace_size)",
                who, w.total);
  if (w.nsplit > 1 || w.blocks > 0) {
    char *ws = (char *)a->workspace;
    p.ws_m = (float *)(ws + w.m_off);
    p.ws_l = (float *)(ws + w.l_off);
    p.ws_o = (float *)(ws + w.o_off);
  }
  p.seen = nullptr;
  p.seen_shift = w.seen_shift;
  p.cuts = w.blocks > 0 ? (int2 *)((char *)a->workspace + w.cuts_off) : nullptr;
  if (mode != PF_ARITH) {
    p.tiles = (uint8_t *)a->workspace;
    if (w.blocks > 0) p.seen = (uint32_t *)((char *)a->workspace + w.seen_off);
    const dim3 cgrid((unsigned)div_up(div_up(a->hot_len, kPfKeys), kMaskTilesPerBlock), (unsigned)div_up(Q, kPfRows),
                     (unsigned)(p.mask_b * p.mask_h));
    if (cgrid.y > 65535 || cgrid.z > 65535) return fail(KIV_ERR_UNSUPPORTED, "%s: too many query rows", who);
    hipLaunchKernelGGL(mask_tiles_kernel, cgrid, dim3(kPfThreads), 0, st, p);
  }
  int rc = with_kt(kt, [&](auto ktc) {
    constexpr int KTV = decltype(ktc)::value;
    if constexpr (KTV == 16) {
      return (int)fail(KIV_ERR_UNSUPPORTED, "%s: head_dim 512 unsupported", who);
    } else {
      const int64_t nblocks = w.blocks > 0 ? w.blocks : div_up(Q, PfShape<KTV>::ROWS) * B * hq * p.nsplit;
      if (nblocks > INT32_MAX) return (int)fail(KIV_ERR_UNSUPPORTED, "%s: too many query rows", who);
      const dim3 grid((unsigned)nblocks);
      auto launch = [&](auto dtc, auto mkc) {
        constexpr int DTV = decltype(dtc)::value, MKV = decltype(mkc)::value;
        if constexpr (KTV <= 4)
          hipLaunchKernelGGL((prefill_attn32_kernel<DTV, KTV, MKV>), grid, dim3(kPfThreads), 0, st, p);
        else
          hipLaunchKernelGGL((prefill_attn_kernel<DTV, KTV, MKV>), grid, dim3(kPfThreads), 0, st, p);
      };
      using std::integral_constant;
      auto by_mode = [&](auto dtc) {
        if (mode == PF_ARITH) launch(dtc, integral_constant<int, PF_ARITH>{});
        else if (mode == PF_BOOL) launch(dtc, integral_constant<int, PF_BOOL>{});
        else launch(dtc, integral_constant<int, PF_FLOAT>{});
      };
      if (dt == KIV_DTYPE_BF16) by_mode(integral_constant<int, DT_BF16>{});
      else by_mode(integral_constant<int, DT_F16>{});
      if (p.nsplit > 1) {
        const int rows_per_block = kPfThreads / (D / 4);
        const dim3 cgrid((unsigned)div_up((int64_t)B * Q * hq, rows_per_block));
        if (dt == KIV_DTYPE_BF16)
          hipLaunchKernelGGL(prefill_combine_kernel<DT_BF16>, cgrid, dim3(kPfThreads), 0, st, p, D);
        else
          hipLaunchKernelGGL(prefill_combine_kernel<DT_F16>, cgrid, dim3(kPfThreads), 0, st, p, D);
      }
      if (w.blocks > 0) {
        const int rows_per_block = kPfThreads / (D / 4);
        const dim3 mgrid((unsigned)div_up(part_rows(Q), rows_per_block), (unsigned)(p.sh.nrb * B * hq));
        if (dt == KIV_DTYPE_BF16)
          hipLaunchKernelGGL(prefill_merge_kernel<DT_BF16>, mgrid, dim3(kPfThreads), 0, st, p, D);
        else
          hipLaunchKernelGGL(prefill_merge_kernel<DT_F16>, mgrid, dim3(kPfThreads), 0, st, p, D);
      }
      return (int)KIV_OK;
    }
  });
  if (rc) return rc;
  KIV_HIP(hipGetLastError());
  return KIV_OK;
}

}  // extern "C"
