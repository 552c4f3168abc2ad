// Sparse MLA decode of many rows (prompt chunks), over the same inputs as
// ekv_decode.hip: gathered latent rows with the per-head attention sink in the
// softmax denominator.
//
// Workgroup = (query row t, block of 32 heads), 4 waves, two workgroups a CU
// (bf16 rows: one).  The row's valid entries go through in steps of 32 cache
// rows; wave w:
//   * scores: S^T = K Q^T of the 32 heads and rows over the 16-dim blocks 4 ks +
//     w (v_mfma_f32_32x32x16_bf16, A = the rows from LDS, fp8 converted exactly
//     to bf16, B = its part of q held in registers); the four waves' sums meet
//     through LDS, wave w taking rows [8 w, +8);
//   * weights: exp2(score - reference), row scale folded in, as a pair of bf16
//     B operands hi = bf16(P), lo = bf16(P - hi), published in LDS.  A head's
//     reference is its maximum over the steps before; a step that exceeds it by
//     more than 8 log2 units (rare after the first steps) moves it and has its
//     weights computed again, so no barrier waits for the maximum and P <= 2^8;
//   * O^T[128 w, +128) += V^T P^T (the same MFMA).
// Two barriers a step; the row loads of the two steps after it are in flight.
// What bounds it: issue (a SIMD issues a conversion or similar VALU
// instruction per 4.5 cycles, and an MFMA costs it about two such slots
// whatever its size) and, of a workgroup alone, the chain scores -> weights ->
// products.  So K and V values are converted once per 32 heads, the products
// use the large MFMA, and the second workgroup of a CU issues while the first
// waits; a row's head blocks run side by side on one XCD and share its rows
// through the L2.
// V^T (channels x entries) is read straight from the row-major row image with
// transposing LDS reads (ds_read_b64_tr_b8 / _b16); S^T's accumulator layout
// is the B-operand layout of P^T, so P is published as it stands.  The hi/lo
// pair carries P to about 2^-16 relative (one bf16 alone is 2^-8, which rows
// of a few entries that nearly cancel expose); V is exact in bf16.
// A prologue resolves every index entry to a cache slot (block table lookup)
// and drops the masked ones (order kept), so a row costs its valid entries.
// Against splits of 32 tiles with fp32 partials and a combine (the few-row
// kernel): 4096 rows of 2176 entries 2.78 -> 2.07 ms, 2331 rows of 2176 of
// which 515 valid on average 1.63 -> 0.39 ms, 6000 rows of about 137 entries
// 0.73 -> 0.40 ms (64 heads, fp8).  4096 rows, by the counters: 4000 cycles a
// pair of 32-row steps on a CU (two workgroups), prologues and epilogues
// included, of which the matrix cores work 1600 (40%).
#include "ekv_decode.h"
#include "ekv_internal.h"

namespace ekv {
namespace decode_rows {

constexpr int kHeadBlock = 32;
constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kMaxEntries = 2176;     // index entries of a row (2048 + 128)
constexpr int kTile = 32;             // cache rows of a step

typedef float f32x16 __attribute__((ext_vector_type(16)));

// Row images hold a step's rows as cached (e4m3fn bytes, or bf16), unpadded,
// with each row's 16-byte chunks permuted (chunk j of row r is stored at
// chunk swz(j, r), an XOR within runs of 8 chunks, of 4 for the last 4 of a
// 36-chunk row) so that the 16 rows a fragment read touches spread over the
// LDS banks.  For 576-byte rows (144 dwords, so rows 4 apart start on the
// same bank) the XOR value is parity(r & 6) | parity(r & 9) << 1 |
// parity(r & 16) << 2, which spreads both the K fragment reads
// (rows 0..31 at one chunk) and the transposed V reads (16 rows at two chunks)
// evenly over the banks.  Rows arrive by direct
// global->LDS loads: lane i of a load instruction writes bytes [16 i, 16 i + 16) of the instruction's 1 KB.
template <int D, bool BF16>
struct DecodeSmem {
  static constexpr int kRowB = BF16 ? 2 * D : D;       // row bytes
  static constexpr int kChunks = kRowB / 16;           // 16-byte chunks per row
  static constexpr int kImgB = kTile * kRowB;          // bytes of one image
  static constexpr int kLoads = kImgB / 1024;          // 1 KB load instructions per step
  static constexpr int kLoadsPerWave = (kLoads + kWaves - 1) / kWaves;
  __align__(16) uint8_t img[3][kImgB];                 // step i in image i % 3
  __align__(16) uint4 sums[kWaves][3][64];             // the other waves' sums of a wave's rows, per lane
  __align__(16) uint4 p[2][2][64];                     // P operands [K step][hi / lo], per lane
  __align__(16) float kscale[3][kTile];                // row scales of step i (fp8), 0 past the last valid entry
  __align__(16) float smax[kHeadBlock][kWaves];        // the waves' maxima; epilogue: their sums of weights
  float fin[kHeadBlock];                               // epilogue: per-head output factor
  int32_t red[64];                                     // the prologue's counts
  __align__(8) int64_t roff[kTile];                    // row offsets of the step loaded next
  int32_t slot[kMaxEntries];                      // the valid entries' cache slots, -1 past the last
};
static_assert(sizeof(DecodeSmem<576, false>) <= 80 * 1024, "two workgroups a CU");
static_assert(sizeof(DecodeSmem<576, true>) <= 160 * 1024, "one workgroup's LDS");

template <int D, bool BF16>
__device__ __forceinline__ int swz_chunk(int j, int r) {
  using SM = DecodeSmem<D, BF16>;
  if constexpr (SM::kChunks % 8 == 0) {
    return j ^ (r & 7);
  } else {
    const int f = (__builtin_popcount(r & 6) & 1) | ((__builtin_popcount(r & 9) & 1) << 1) |
                  ((__builtin_popcount(r & 16) & 1) << 2);
    return j < 32 ? (j ^ f) : (32 + ((j - 32) ^ (f & 3)));
  }
}

// Byte offset in a tile image of bytes [8 h, 8 h + 8) of 16-byte chunk c of row r.
template <int D, bool BF16>
__device__ __forceinline__ int img_off(int r, int c, int h) {
  return r * DecodeSmem<D, BF16>::kRowB + 16 * swz_chunk<D, BF16>(c, r) + 8 * h;
}

// Image offsets of this lane's K fragments: 8 dims of row r at K step ks, the
// block 4 ks + w of 16 dims, half hl of it.  Runs of 8 chunks are 128 bytes
// apart, so all steps read from a few bases (fp8: chunk 4 ks + w at
// off[ks % 2] + 128 (ks / 2), and that of the last four chunks of a 36-chunk
// row at off[2]; bf16: chunk 8 ks + 2 w + hl at off[0] + 128 ks).
template <int D, bool BF16>
struct KeyLanes {
  static constexpr int kN = BF16 ? 1 : (DecodeSmem<D, BF16>::kChunks % 8 == 0 ? 2 : 3);
  uint32_t off[kN];
};

template <int D, bool BF16>
__device__ __forceinline__ KeyLanes<D, BF16> key_lanes(int r, int w, int hl) {
  KeyLanes<D, BF16> kl;
#pragma unroll
  for (int i = 0; i < KeyLanes<D, BF16>::kN; ++i) {
    if constexpr (BF16) kl.off[i] = img_off<D, BF16>(r, 2 * w + hl, 0);
    else kl.off[i] = img_off<D, BF16>(r, (i < 2 ? 4 * i : 32) + w, hl);
  }
  return kl;
}

// Max of v over the lanes l and l ^ 32, with a VALU lane swap instead of an
// LDS permute: after a swap of the halves between two copies of v, the max of
// the two results is the pairwise max in every lane.
__device__ __forceinline__ float max_halves(float v) {
  const uint32_t w = __float_as_uint(v);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// Row (of 16) of k-slot m (0..7) of half-wave hl in the S^T accumulators / the
// V^T P^T operands.
__device__ __forceinline__ int slot_row(int hl, int m) { return m < 4 ? 4 * hl + m : 8 + 4 * hl + (m - 4); }

// ---------------------------------------------------------------------------
// Row loads.  Instruction k of a step covers image bytes [1024 k,
// 1024 k + 1024); lane i its 16-byte chunk 64 k + i, i.e. row
// (64 k + i) / kChunks, stored chunk j = (64 k + i) % kChunks, which holds
// row chunk swz(j, r).  Rows past the last valid entry load cache row 0
// (zeroed once the step has landed).  Wave w issues the instructions
// k = w + 4 j; this lane then copies byte col[j] on of step entry row[j].
template <int D, bool BF16>
struct TileLanes {
  static constexpr int kN = DecodeSmem<D, BF16>::kLoadsPerWave;
  int row[kN], col[kN];
};

template <int D, bool BF16>
__device__ __forceinline__ TileLanes<D, BF16> tile_lanes(int w) {
  using SM = DecodeSmem<D, BF16>;
  const int lane = threadIdx.x & 63;
  TileLanes<D, BF16> tl;
#pragma unroll
  for (int j = 0; j < SM::kLoadsPerWave; ++j) {
    const int pos = (w + kWaves * j) * 64 + lane;
    const int r = min(pos / SM::kChunks, kTile - 1), jj = pos % SM::kChunks;  // (past kLoads: not issued)
    tl.row[j] = r;
    tl.col[j] = 16 * swz_chunk<D, BF16>(jj, r);
  }
  return tl;
}

// Byte offset of a slot's row in the cache (-1: that of slot 0).
template <int D, bool BF16>
__device__ __forceinline__ int64_t row_offset(const DecodeArgs& a, int slot) {
  const int64_t s = max(slot, 0);
  if constexpr (BF16) return s * (2 * D);
  else return (s >> 6) * a.page_stride + (s & 63) * D;
}

template <int D, bool BF16>
__device__ __forceinline__ void issue_row(const DecodeArgs& a, int w, int j, int64_t off, uint8_t* img) {
  using SM = DecodeSmem<D, BF16>;
  const int k = w + kWaves * j;
  if ((j + 1) * kWaves > SM::kLoads && k >= SM::kLoads) return;  // (wave-uniform)
  load_lds16(a.cache + off, img + 1024 * k);
}

// The row scales of a step (fp8), by one wave: lane i's row i, of slot `slot`.
template <int D, bool BF16>
__device__ __forceinline__ void issue_scales(const DecodeArgs& a, DecodeSmem<D, BF16>& sm, int slot, int tile) {
  if constexpr (!BF16) {
    if ((threadIdx.x & 63) >= kTile) return;
    const int64_t s = max(slot, 0);
    load_lds4(a.cache + (s >> 6) * a.page_stride + kPageTokens * D + (s & 63) * 4,
              reinterpret_cast<uint8_t*>(sm.kscale[tile % 3]));
  }
}

// Zero the image rows and scales past the last valid entry of a step whose
// loads by this wave have landed (the split's last step; a weight of 0 times
// an infinity or NaN of whatever row was loaded there would not be 0).
template <int D, bool BF16>
__device__ __forceinline__ void zero_masked(DecodeSmem<D, BF16>& sm, const TileLanes<D, BF16>& tl, int w, int tile) {
  using SM = DecodeSmem<D, BF16>;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < SM::kLoadsPerWave; ++j) {
    const int k = w + kWaves * j;
    if (k >= SM::kLoads) break;
    if (sm.slot[tile * kTile + tl.row[j]] < 0)
      *reinterpret_cast<uint4*>(sm.img[tile % 3] + 1024 * k + 16 * lane) = make_uint4(0, 0, 0, 0);
  }
  if (w == kWaves - 1 && lane < kTile && sm.slot[tile * kTile + lane] < 0) sm.kscale[tile % 3][lane] = 0.0f;
}

// ---------------------------------------------------------------------------
// This lane's V^T fragment (32 channels from 128 w + 32 c on x the 16 rows of
// K step kq), read transposed from the row-major image: 8 fp8 bytes (in .x,
// .y) or 8 bf16 values, rows slot_row(lane / 32, m) of channel lane % 32.
template <int D, bool BF16>
__device__ __forceinline__ uint4 pv_read(const uint8_t* img, int kq, int w, int c) {
  const int lane = threadIdx.x & 63;
  const int hl = lane >> 5, i = lane & 15;
  const int ch = 128 * w + 32 * c + 16 * ((lane >> 4) & 1);
  const uint8_t* base = img;
  const int r0 = 16 * kq;
  if constexpr (BF16) {
    const int cl = ch + 4 * (i & 3);
    const i16x4 lo =
        lds_read_tr16(base + img_off<D, BF16>(r0 + slot_row(hl, i >> 2), cl >> 3, (cl >> 2) & 1));
    const i16x4 hi =
        lds_read_tr16(base + img_off<D, BF16>(r0 + slot_row(hl, 4 + (i >> 2)), cl >> 3, (cl >> 2) & 1));
    const i16x4 both[2] = {lo, hi};
    return __builtin_bit_cast(uint4, both);
  } else {
    const uint2 v = lds_read_tr8(base + img_off<D, BF16>(r0 + slot_row(hl, i >> 1), ch >> 4, i & 1));
    return make_uint4(v.x, v.y, 0u, 0u);
  }
}

template <bool BF16>
__device__ __forceinline__ bf16x8 pv_frag(const uint4& raw) {
  if constexpr (BF16) return __builtin_bit_cast(bf16x8, raw);
  else return fp8x8_bf16(make_uint2(raw.x, raw.y));
}

// Eight channels of head h times f as bf16: from c0 on for the lower
// half-wave, c0 + 8 for the upper one.  v holds accumulator values i, i + 4
// (channels c0 + 4 hl + i and c0 + 8 + 4 hl + i): the halves swap a group of
// four each.
__device__ __forceinline__ void store_o(const DecodeArgs& a, int t, int h, int c0, float f, const float (&v)[8]) {
  const int hl = (threadIdx.x & 63) >> 5;
  uint32_t g[2][2];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int e = 0; e < 2; ++e)
      g[k][e] = static_cast<uint32_t>(f32_to_bf16(v[4 * k + 2 * e] * f)) |
                (static_cast<uint32_t>(f32_to_bf16(v[4 * k + 2 * e + 1] * f)) << 16);
  const auto x = __builtin_amdgcn_permlane32_swap(g[0][0], g[1][0], false, false);
  const auto y = __builtin_amdgcn_permlane32_swap(g[0][1], g[1][1], false, false);
  if (h < a.heads)
    *reinterpret_cast<uint4*>(a.out + static_cast<int64_t>(t) * a.out_tok_stride + h * a.out_head_stride + c0 + 8 * hl) =
        make_uint4(x[0], y[0], x[1], y[1]);
}

// ---------------------------------------------------------------------------
template <int D, bool BF16>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
sparse_decode_rows_kernel(DecodeArgs a) {
  extern __shared__ __align__(16) uint8_t smem_raw[];
  using SM = DecodeSmem<D, BF16>;
  SM& sm = *reinterpret_cast<SM*>(smem_raw);
  constexpr int KS = D / (16 * kWaves);  // K steps of a wave
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, col = lane & 31;

  // An XCD (b % 8) takes a run of rows, the head blocks of a row next to each
  // other.
  const int b = blockIdx.x;
  const int hbs = (a.heads + kHeadBlock - 1) / kHeadBlock;  // 1 or 2
  const int hb = hbs > 1 ? (b / kXcds) & 1 : 0;
  const int per_xcd = (a.rows + kXcds - 1) / kXcds;
  const int t = (b % kXcds) * per_xcd + b / kXcds / hbs;
  if (t >= a.rows) return;
  const int head = kHeadBlock * hb + col;  // the head of this lane's scores, weights and outputs
  const bool has_head = head < a.heads;

  // Prologue: entries -> slots (index, then block table), each gather issued
  // for all of the thread's entries before the next.
  constexpr int kPrologue = (kMaxEntries + kThreads - 1) / kThreads;
  int64_t sv[kPrologue];
  const int len = row_len(a, t);
#pragma unroll
  for (int j = 0; j < kPrologue; ++j) {
    const int e = tid + kThreads * j;
    sv[j] = (e < len) ? a.indices[static_cast<int64_t>(t) * a.idx_stride + e] : -1;
  }
  if (a.block_table != nullptr) {
    const int32_t* bt = a.block_table + static_cast<int64_t>(a.req_ids[t]) * a.bt_stride;
#pragma unroll
    for (int j = 0; j < kPrologue; ++j) {
      const int64_t idx = sv[j];
      const bool ok = idx >= 0 && (idx >> 6) < a.bt_stride;
      const int64_t page = bt[ok ? (idx >> 6) : 0];
      sv[j] = ok ? page * kPageTokens + (idx & 63) : -1;
    }
  }
  // Valid entries to consecutive positions, in order: (batch j, wave) counts,
  // scanned by every wave.
  constexpr int kCounts = kPrologue * kWaves;
  static_assert(kCounts <= 64, "one lane per count");
  uint64_t bal[kPrologue];
#pragma unroll
  for (int j = 0; j < kPrologue; ++j) {
    bal[j] = __ballot(sv[j] >= 0 && sv[j] < a.num_rows);
    if (lane == 0) sm.red[j * kWaves + wave] = static_cast<int>(__popcll(bal[j]));
  }
  __syncthreads();
  int cnts = lane < kCounts ? sm.red[lane] : 0;
  const int own = cnts;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(cnts, off);
    if (lane >= off) cnts += y;
  }
  const int nvalid = __builtin_amdgcn_readfirstlane(__shfl(cnts, 63));
  cnts -= own;
  const int ntiles = (nvalid + kTile - 1) / kTile;
  const int e_pad = ntiles * kTile;
#pragma unroll
  for (int j = 0; j < kPrologue; ++j) {
    const int base = __shfl(cnts, j * kWaves + wave);
    if ((bal[j] >> lane) & 1)
      sm.slot[base + static_cast<int>(__popcll(bal[j] & ((uint64_t{1} << lane) - 1)))] = static_cast<int32_t>(sv[j]);
  }
  if (tid < kTile && nvalid + tid < e_pad) sm.slot[nvalid + tid] = -1;
  const bool ragged = nvalid < e_pad;
  __syncthreads();
  // Steps 0 and 1 and q requested together.
  const TileLanes<D, BF16> tl = tile_lanes<D, BF16>(wave);
  auto issue_step = [&](int tile) {
    int sl[SM::kLoadsPerWave];
#pragma unroll
    for (int j = 0; j < SM::kLoadsPerWave; ++j) sl[j] = sm.slot[tile * kTile + tl.row[j]];
#pragma unroll
    for (int j = 0; j < SM::kLoadsPerWave; ++j)
      issue_row<D, BF16>(a, wave, j, row_offset<D, BF16>(a, sl[j]) + tl.col[j], sm.img[tile % 3]);
    if (wave == kWaves - 1) issue_scales<D, BF16>(a, sm, sm.slot[tile * kTile + col], tile);
  };
  if (ntiles > 0) issue_step(0);
  if (ntiles > 1) issue_step(1);
  bf16x8 qb[KS];  // B operand of S^T = K Q^T: head `head`, dims 16 (4 ks + w) + 8 hl .. +7
  {
    // (a head past the call's reads head 0; its scores are not used)
    const uint16_t* qrow = a.q + static_cast<int64_t>(t) * a.q_tok_stride + (has_head ? head : 0) * a.q_head_stride;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qb[ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(qrow + 16 * (4 * ks + wave) + 8 * hl));
  }
  const float sink = (a.sinks != nullptr && has_head) ? a.sinks[head] * kLog2e : -INFINITY;
  wait_vm<0>();
  if (ragged && ntiles <= 2) zero_masked<D, BF16>(sm, tl, wave, ntiles - 1);
  __syncthreads();

  KeyLanes<D, BF16> kl = key_lanes<D, BF16>(col ^ (8 * wave), wave, hl);
  f32x16 o[4];  // O^T[128 w + 32 c + ...][head]
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[c][i] = 0.0f;
  float mref = -INFINITY;  // the head's reference (log2 units), the same in every wave
  float lsum = 0.0f;       // this lane's share of the head's l
  const float sc2 = a.scale * kLog2e;
  // The head's maximum over a step's rows.
  auto step_max = [&]() -> float {
    const float4 m = *reinterpret_cast<const float4*>(sm.smax[col]);
    return fmaxf(fmaxf(m.x, m.y), fmaxf(m.z, m.w));
  };
  // The reference moves to mx where that is larger; the factor of what was
  // accumulated before.
  auto move_ref = [&](float mx) -> float {
    const float mnew = fmaxf(mref, mx);
    float al = 1.0f;
    if (mnew != -INFINITY) {
      al = (mref == -INFINITY) ? 0.0f : exp2f(mref - mnew);
      mref = mnew;
    }
    return al;
  };
  auto scale_o = [&](float al) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[c][i] *= al;
  };
  float x[4], ksx[4];  // this lane's scores of a step: rows 8 wave + 4 hl + i
  float psum = 0.0f;
  // The weights of the scores x, published as the step's operands.
  auto weights = [&] {
    const bool live = mref != -INFINITY;
    psum = 0.0f;
    uint32_t hi[2], lo[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      float w[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float p = live ? __builtin_amdgcn_exp2f(x[2 * m + e] - mref) : 0.0f;  // (tiny weights flush to 0)
        psum += p;
        w[e] = p * ksx[2 * m + e];
      }
      hi[m] = bf16x2_bits(w[0], w[1]);
      const float h0 = __uint_as_float(hi[m] << 16), h1 = __uint_as_float(hi[m] & 0xffff0000u);
      lo[m] = bf16x2_bits(w[0] - h0, w[1] - h1);  // exact differences
    }
    // rows 8 wave + 4 hl + i are k-slots 4 (wave % 2) + i of K step wave / 2
    reinterpret_cast<uint2*>(&sm.p[wave >> 1][0][lane])[wave & 1] = make_uint2(hi[0], hi[1]);
    reinterpret_cast<uint2*>(&sm.p[wave >> 1][1][lane])[wave & 1] = make_uint2(lo[0], lo[1]);
  };

  uint4 kr[KS];  // K fragments of the step to score next
  auto read_k = [&](int s) {
    const uint8_t* imgs = reinterpret_cast<const uint8_t*>(sm.img);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if constexpr (BF16) {
        kr[ks] = *reinterpret_cast<const uint4*>(imgs + kl.off[0] + 128 * ks);
      } else {
        const uint2 v = *reinterpret_cast<const uint2*>(
            ks < 8 ? imgs + kl.off[ks & 1] + 128 * (ks >> 1) : imgs + kl.off[KeyLanes<D, BF16>::kN - 1]);
        kr[ks] = make_uint4(v.x, v.y, 0u, 0u);
      }
    }
    const uint32_t move = s % 3 == 2 ? 0u - 2 * SM::kImgB : SM::kImgB;  // on to the next step's image
#pragma unroll
    for (int i = 0; i < KeyLanes<D, BF16>::kN; ++i) kl.off[i] += move;
  };
  if (!BF16 && ntiles > 0) read_k(0);
  for (int s = 0; s < ntiles; ++s) {
    const uint8_t* img = sm.img[s % 3];
    if (BF16) read_k(s);  // (no registers for it earlier)
    // Scores.  Accumulator rows [8 j, +8) are the image's rows [8 (j ^ wave), +8),
    // so a wave keeps the first of them.
    f32x16 st;
#pragma unroll
    for (int i = 0; i < 16; ++i) st[i] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pv_frag<BF16>(kr[ks]), qb[ks], st, 0, 0, 0);
#pragma unroll
    for (int j = 1; j < kWaves; ++j)
      sm.sums[wave ^ j][j - 1][lane] =
          make_uint4(__float_as_uint(st[4 * j]), __float_as_uint(st[4 * j + 1]), __float_as_uint(st[4 * j + 2]),
                     __float_as_uint(st[4 * j + 3]));
    __syncthreads();  // (and step s - 1's products are done with its image and operands)

    // The row offsets of step s + 2, by the last wave; the loads go out
    // between the products.  (Worked out once per row: per load, the 64-bit
    // multiplies took a quarter of the step.)
    const bool load = s + 2 < ntiles;
    int next_slot = 0;
    if (load && wave == kWaves - 1) {
      next_slot = sm.slot[(s + 2) * kTile + col];
      if (hl == 0) sm.roff[col] = row_offset<D, BF16>(a, next_slot);
    }
    {
      uint4 other[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) other[j] = sm.sums[wave][j][lane];
      float4 k4 = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
      if constexpr (!BF16) k4 = *reinterpret_cast<const float4*>(&sm.kscale[s % 3][8 * wave + 4 * hl]);
      const float kv[4] = {k4.x, k4.y, k4.z, k4.w};
      const uint32_t ov[3][4] = {{other[0].x, other[0].y, other[0].z, other[0].w},
                                 {other[1].x, other[1].y, other[1].z, other[1].w},
                                 {other[2].x, other[2].y, other[2].z, other[2].w}};
      float mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = (st[i] + __uint_as_float(ov[0][i])) + (__uint_as_float(ov[1][i]) + __uint_as_float(ov[2][i]));
        const bool ok = BF16 ? s * kTile + 8 * wave + 4 * hl + i < nvalid : kv[i] > 0.0f;
        ksx[i] = BF16 ? (ok ? 1.0f : 0.0f) : kv[i];
        x[i] = ok ? v * (sc2 * kv[i]) : -INFINITY;
        mx = fmaxf(mx, x[i]);
      }
      mx = max_halves(mx);
      sm.smax[col][wave] = mx;  // (both halves, the same value)
    }
    if (s == 0) {  // the first reference
      __syncthreads();
      move_ref(step_max());
    }
    weights();
    constexpr int kRaw = BF16 ? 1 : 2;  // (bf16 fragments take twice the registers)
    uint4 raw[kRaw][4], pr[2][2];
    if constexpr (!BF16) {
#pragma unroll
      for (int c = 0; c < 4; ++c) raw[0][c] = pv_read<D, BF16>(img, 0, wave, c);
    }
    wait_vm<0>();  // this wave's loads of step s + 1
    if (ragged && s > 0 && s + 2 == ntiles) zero_masked<D, BF16>(sm, tl, wave, s + 1);
    __syncthreads();

    // Products, and the step's maximum against the reference it used.
    auto read_p = [&] {
#pragma unroll
      for (int kq = 0; kq < 2; ++kq) {
        pr[kq][0] = sm.p[kq][1][lane];
        pr[kq][1] = sm.p[kq][0][lane];
      }
    };
    read_p();
    int64_t ro[SM::kLoadsPerWave];
    if (load) {
#pragma unroll
      for (int j = 0; j < SM::kLoadsPerWave; ++j) ro[j] = sm.roff[tl.row[j]];
    }
    const float mx = step_max();
    if (__any(mx > mref + kRescaleSlack)) {  // the same in every wave (also a first finite maximum)
      const float al = move_ref(mx);
      scale_o(al);
      lsum *= al;
      weights();
      __syncthreads();
      read_p();
    }
    lsum += psum;
#pragma unroll
    for (int c = 0; c < 4; ++c) raw[kRaw - 1][c] = pv_read<D, BF16>(img, kRaw - 1, wave, c);
    if (!BF16 && s + 1 < ntiles) read_k(s + 1);
#pragma unroll
    for (int kq = 0; kq < 2; ++kq) {
      bf16x8 v[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        v[c] = pv_frag<BF16>(raw[kq % kRaw][c]);
        if (kRaw == 1 && kq == 0) raw[0][c] = pv_read<D, BF16>(img, 1, wave, c);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v[c], __builtin_bit_cast(bf16x8, pr[kq][e]), o[c], 0, 0, 0);
        // a few of the loads at a time: a burst holds up the wave that issues it
        constexpr int kPer = (SM::kLoadsPerWave + 3) / 4;
        if (load) {
#pragma unroll
          for (int j = kPer * (2 * kq + e); j < kPer * (2 * kq + e + 1) && j < SM::kLoadsPerWave; ++j)
            issue_row<D, BF16>(a, wave, j, ro[j] + tl.col[j], sm.img[(s + 2) % 3]);
          if (kq == 1 && e == 1 && wave == kWaves - 1) issue_scales<D, BF16>(a, sm, next_slot, s + 2);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // Epilogue: the waves' sums of weights meet, wave 0 finishes the heads'
  // softmax (the sink, the lse) and publishes the output factors.
  const float lw = lsum + __shfl_xor(lsum, 32);
  __syncthreads();  // (the last step's maxima have been read)
  sm.smax[col][wave] = lw;
  __syncthreads();
  if (wave == 0 && hl == 0 && has_head) {
    const float4 l4 = *reinterpret_cast<const float4*>(sm.smax[col]);
    const float lt = (l4.x + l4.y) + (l4.z + l4.w);
    float den = lt, numf = 1.0f;
    if (a.sinks != nullptr) {
      const float mp = fmaxf(mref, sink);
      if (mp != -INFINITY) {
        numf = (mref == -INFINITY) ? 0.0f : exp2f(mref - mp);
        den = lt * numf + exp2f(sink - mp);
      }
    }
    if (a.lse != nullptr)
      a.lse[static_cast<int64_t>(t) * a.lse_stride + head] = (lt > 0.0f) ? (mref + log2f(lt)) * kLn2 : -INFINITY;
    sm.fin[col] = (den > 0.0f) ? numf / den : 0.0f;
  }
  __syncthreads();
  const float f = has_head ? sm.fin[col] : 0.0f;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const float v[8] = {o[c][8 * k],     o[c][8 * k + 1], o[c][8 * k + 2], o[c][8 * k + 3],
                          o[c][8 * k + 4], o[c][8 * k + 5], o[c][8 * k + 6], o[c][8 * k + 7]};
      store_o(a, t, head, 128 * wave + 32 * c + 16 * k, f, v);
    }
}

template <int D, bool BF16>
void launch(const DecodeArgs& a, hipStream_t s) {
  const size_t smem = sizeof(DecodeSmem<D, BF16>);
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(sparse_decode_rows_kernel<D, BF16>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
  const int64_t per_xcd = (a.rows + kXcds - 1) / kXcds;
  const dim3 grid(static_cast<uint32_t>(kXcds * per_xcd * ((a.heads + kHeadBlock - 1) / kHeadBlock)));
  hipLaunchKernelGGL((sparse_decode_rows_kernel<D, BF16>), grid, dim3(kThreads), smem, s, a);
}

}  // namespace decode_rows

// The line between this kernel (a whole row a workgroup: about 9 us + 1.35 us
// per 32 entries, no partials) and the few-row one (rows split over the CUs,
// then a combine), measured at 1..640 rows of full index rows of 33..2176
// entries, 16 / 32 / 48 / 64 heads, both widths and cache types.  Ratios are
// the few-row kernel's time over this one's.
//   * fp8 caches, two workgroups a CU.  From 192 rows on no splitting is needed
//     to fill the CUs (64 heads, 2176 entries: 192 rows 1.30, 256: 1.68; the
//     least from there on 1.01, 48 heads).
//   * Short rows: the combine costs more than the splits give (64 heads, 256
//     entries: 1 row 1.11, 64 rows 1.63; 384: 8 rows 0.99, 16 rows 1.23; 48
//     heads, 2 rows: 192 entries 1.06, 256 0.96; 32 heads, 8 rows: 192 1.13, 256
//     0.97).
//   * 33..64 heads, 96..128 rows: two workgroups of a row fill the CUs (64 heads,
//     128 rows: 2176 entries 1.17, 768 1.12).  The few-row kernel runs its
//     workgroups at once while they number at most 256, and is the faster one
//     for long rows up to there (48 heads, 1152 entries: 120 rows 0.94, 128 rows
//     1.56).  Up to 191 rows while running two a CU pays (64 heads: 160 rows of
//     1152 1.32, of 2176 0.96).
//   * bf16 caches: the row images leave room for one workgroup a CU, so rows
//     above 32 heads, two workgroups each, fill the CUs once at 128 rows (64
//     heads, 192 entries: 128 rows 1.64, 136 rows 0.82; 2048 rows of 2176 0.83)
//     and the gain per row is smaller (64 heads, 8 rows: 192 entries 1.20, 320
//     1.00; 48 heads, 2 rows: 192 0.99, 256 0.89, 104 rows: 512 1.04, 1800
//     1.24, 2176 0.92).  Up to 32 heads: from 192 rows on, but not where a
//     second round of long rows is mostly empty (32 heads, 288 rows: 768
//     entries 1.04, 2176 0.87; 384 rows of 2176 1.08).
// Rows past what the LDS holds slots for take the few-row kernel.
bool decode_rows_takes(int32_t num_tokens, int32_t heads, int32_t width, bool cache_bf16, int64_t split_groups) {
  if (width > decode_rows::kMaxEntries || num_tokens >= (1 << 28)) return false;
  if (heads <= 32) {
    if (num_tokens < 192) return width <= 192;
    return !cache_bf16 || num_tokens <= 256 || num_tokens >= 384 || width <= 768;
  }
  const bool split_rounds = split_groups > 256;  // the few-row kernel's workgroups do not all run at once
  if (cache_bf16) {
    if (num_tokens > 128) return false;
    return width <= 192 || (width <= 320 && num_tokens >= 16) ||
           (num_tokens >= 96 && (width <= 512 || (split_rounds && width <= 1800)));
  }
  if (num_tokens >= 192) return true;
  if (num_tokens > 128) return width <= 1152;
  return width <= (heads > 48 || num_tokens >= 8 ? 256 : 192) || (width <= 384 && num_tokens >= 16) ||
         (num_tokens >= 96 && (width <= 768 || split_rounds));
}

int launch_decode_rows(const DecodeArgs& a, int32_t dim, bool cache_bf16, hipStream_t s) {
  if (dim == 576) {
    if (cache_bf16) decode_rows::launch<576, true>(a, s);
    else decode_rows::launch<576, false>(a, s);
  } else {
    if (cache_bf16) decode_rows::launch<512, true>(a, s);
    else decode_rows::launch<512, false>(a, s);
  }
  return ekv_launch_status();
}

}  // namespace ekv
