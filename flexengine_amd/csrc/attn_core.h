// Per-wave paged-attention tile engine shared by the decode and prefill kernels.
//
// A wave owns up to 16 "columns" n (decode: the G query heads of one KV head;
// prefill: 16 query rows of one query head) and walks 16-token key tiles of one
// sequence's paged K/V.  Lane l = 16g + n.
//
//   S^T[16 keys x 16 cols] = K[16 x D] . Q^T[D x 16]        (MFMA 16x16x16 f16)
//     A = K: lane (g,n) loads key n of the tile, 16-byte chunks 4s+g (s < D/32),
//            straight from the pool; each chunk feeds two MFMAs.
//     B = Q: lane (g,n) holds column n's query vector, same chunks.
//     -> lane (g,n) holds the scores of column n for keys 4g..4g+3.
//   online softmax in base 2 (scores scaled by scale*log2(e)); column n's
//     running max is shared by its four lanes (g = 0..3) via two xor-shuffles.
//   O^T[D x 16 cols] += V^T[D x 16 keys] . P^T[16 keys x 16 cols]  (D/16 MFMAs)
//     B = P^T is the score layout above, converted to fp16.
//     A = V^T: V rows are loaded with coalesced 16-byte loads (16 lanes per
//            256-byte row), staged in a per-wave LDS tile with a padded pitch
//            and read back column-wise.
//     -> lane (g,n) accumulates O[col n][d = 16x + 4g + i], so the softmax
//        rescale of column n never leaves the lane.
#pragma once

#include "fe_common.h"

namespace fe {

constexpr int kTile = 16;

template <int D>
struct TileCfg {
  static constexpr int NK = D / 32;       // K chunk loads per lane per tile (= V loads)
  static constexpr int NX = D / 16;       // PV output tiles of 16 dims
  static constexpr int CPR = D / 8;       // 16-byte chunks per K/V row
  static constexpr int RPI = kWave / CPR; // V rows covered by one load instruction
  // LDS pitch of a staged V row: D halves + 32 bytes = D/2 + 8 dwords, which is
  // 8 mod 32 for D = 64 and 128.  The transposing read of a 16-dim slice (see
  // softmax_pv_tile) has each 16-lane group fetch 8 bytes from 4 rows x 4
  // consecutive 8-byte columns; rows 8 dwords apart put those 16 fetches on
  // distinct bank pairs.
  static constexpr int ROWB = D * 2 + 32;
  static constexpr int STAGE = kTile * ROWB;
};

__device__ __forceinline__ int clamp_block(int blk, int nb) {
  return blk < 0 ? 0 : (blk >= nb ? nb - 1 : blk);
}

__device__ __forceinline__ void compiler_fence() { asm volatile("" ::: "memory"); }

// Running-max slack of the online softmax, in base-2 units: the max a tile's
// scores are exponentiated against is only raised when some column's tile max
// exceeds it by more than this, so most tiles skip the rescale of o and l, and
// every probability stays <= 2^kRescaleSlack (exact in fp16 for the PV MFMA).
constexpr float kRescaleSlack = 8.f;

typedef short s16x4 __attribute__((ext_vector_type(4)));

// Shared softmax + PV step of one 16-key tile (scores already in sacc).
// Lane (g,n): sacc[i] = raw score of key t0 + 4g + i for column n; keys at or
// past `limit` are masked.  V rows of the tile are in `stage` (row pitch ROWB).
//
// The PV product O^T[16 dims x 16 cols] += V^T . P^T takes its A operand
// (lane (g,n): V[key 4g+i][dim 16x+n], i = 0..3) from one transposing LDS read
// per 16-dim slice: ds_read_b64_tr_b16 returns to lane l of a 16-lane group
// the halves M[4j + l/4][l%4] (j = 0..3), M[r] being the 8 bytes addressed by
// lane r of the group; lane (g, r) therefore addresses
// V[key 4g + r/4][dims 16x + 4(r%4) .. +3].
template <int D, class E = Fp16>
__device__ __forceinline__ void softmax_pv_tile(f32x4 sacc, int t0, int limit, float scale_log2,
                                                const unsigned char* stage, float& m_run,
                                                float& l_run, f32x4 (&o)[TileCfg<D>::NX]) {
  using C = TileCfg<D>;
  const int lane = lane_id();
  const int g = lane >> 4;
  const int n = lane & 15;
  float sv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int tok = t0 + 4 * g + i;
    sv[i] = tok < limit ? sacc[i] * scale_log2 : kNegInf;
  }
  float mx = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
  mx = fmaxf(mx, shfl_xor_f(mx, 16));
  mx = fmaxf(mx, shfl_xor_f(mx, 32));
  if (__ballot(mx > m_run + kRescaleSlack)) {  // wave-uniform
    const float m_new = fmaxf(m_run, mx);
    const float alpha = m_new == kNegInf ? 1.f : exp2_fast(m_run - m_new);
    l_run *= alpha;
#pragma unroll
    for (int x = 0; x < C::NX; ++x) o[x] *= alpha;
    m_run = m_new;
  }
  const float m_use = m_run == kNegInf ? 0.f : m_run;
  float p[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = exp2_fast(sv[i] - m_use);
  l_run += (p[0] + p[1]) + (p[2] + p[3]);
  const f16x4 pb = to16x4<E>(p[0], p[1], p[2], p[3]);
  const unsigned char* vb = stage + (4 * g + (n >> 2)) * C::ROWB + (n & 3) * 8;
#pragma unroll
  for (int x = 0; x < C::NX; ++x) {
    const s16x4 raw = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(vb + 32 * x));
    o[x] = mma16<E>(__builtin_bit_cast(f16x4, raw), pb, o[x]);
  }
}

template <int D, class E = Fp16>
struct TileCore {
  using C = TileCfg<D>;

  // sequence / pool geometry
  f16* k_pool;
  f16* v_pool;
  const int32_t* trow;  // block-table row of the sequence
  int64_t rs;           // elements per pool row (kv_heads * D)
  int hoff;             // kv_head * D
  int W, NB, BS, bs_log2;
  int tok_end;          // keys >= tok_end are never read
  int limit;            // this lane's column accepts keys < limit
  float scale_log2;
  // optional fused page write of the decode token (position new_pos)
  const f16* knew_row;
  const f16* vnew_row;
  int new_pos;          // -1: none

  unsigned char* stage; // per-wave LDS tile, C::STAGE bytes

  f16x8 qv[C::NK];
  float m_run;
  float l_run;
  f32x4 o[C::NX];

  __device__ __forceinline__ int64_t pool_row(int tok) const {
    int page = tok >> bs_log2;
    page = page < W ? page : W - 1;
    const int blk = clamp_block(trow[page], NB);
    return (int64_t)blk * BS + (tok & (BS - 1));
  }

  __device__ __forceinline__ void init_acc() {
    m_run = kNegInf;
    l_run = 0.f;
#pragma unroll
    for (int x = 0; x < C::NX; ++x) o[x] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  __device__ __forceinline__ void load_tile(int t, f16x8 (&kk)[C::NK], f16x8 (&vv)[C::NK]) const {
    const int lane = lane_id();
    const int g = lane >> 4;
    const int n = lane & 15;
    const int t0 = t * kTile;
    {
      const int tk = t0 + n;
      const int tkc = tk < tok_end ? tk : tok_end - 1;
      f16* kp = k_pool + pool_row(tkc) * rs + hoff;
      if (tk == new_pos) {
#pragma unroll
        for (int s = 0; s < C::NK; ++s) {
          kk[s] = ld16(knew_row + (4 * s + g) * 8);
          st16(kp + (4 * s + g) * 8, kk[s]);
        }
      } else {
#pragma unroll
        for (int s = 0; s < C::NK; ++s) kk[s] = ld16(kp + (4 * s + g) * 8);
      }
    }
    const int cv = lane % C::CPR;
#pragma unroll
    for (int j = 0; j < C::NK; ++j) {
      const int tv = t0 + j * C::RPI + lane / C::CPR;
      const bool ok = tv < tok_end;
      const int tvc = ok ? tv : tok_end - 1;
      f16* vp = v_pool + pool_row(tvc) * rs + hoff + cv * 8;
      f16x8 val;
      if (tv == new_pos) {
        val = ld16(vnew_row + cv * 8);
        st16(vp, val);
      } else {
        val = ld16(vp);
      }
      vv[j] = ok ? val : f16x8{};
    }
  }

  __device__ __forceinline__ void compute_tile(int t, const f16x8 (&kk)[C::NK],
                                               const f16x8 (&vv)[C::NK]) {
    const int lane = lane_id();
    const int t0 = t * kTile;
    f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < C::NK; ++s) {
      sacc = mma16<E>(lo4(kk[s]), lo4(qv[s]), sacc);
      sacc = mma16<E>(hi4(kk[s]), hi4(qv[s]), sacc);
    }
    // stage the V rows of this tile (row-major, padded pitch)
    compiler_fence();
    {
      const int cv = lane % C::CPR;
#pragma unroll
      for (int j = 0; j < C::NK; ++j) {
        const int r = j * C::RPI + lane / C::CPR;
        unsigned char* dst = stage + r * C::ROWB + cv * 16;
        *reinterpret_cast<f16x8*>(dst) = vv[j];  // ROWB is a multiple of 16
      }
    }
    compiler_fence();
    softmax_pv_tile<D, E>(sacc, t0, limit, scale_log2, stage, m_run, l_run, o);
    compiler_fence();
  }

  // Tiles t_first, t_first + step, ... < t_end with one tile of prefetch.
  __device__ __forceinline__ void run(int t_first, int step, int t_end) {
    f16x8 ka[C::NK], va[C::NK], kb[C::NK], vb[C::NK];
    int t = t_first;
    if (t < t_end) load_tile(t, ka, va);
    while (t < t_end) {
      if (t + step < t_end) load_tile(t + step, kb, vb);
      compute_tile(t, ka, va);
      t += step;
      if (t >= t_end) break;
      if (t + step < t_end) load_tile(t + step, ka, va);
      compute_tile(t, kb, vb);
      t += step;
    }
  }

  // Softmax denominator of column n summed over the four lanes g.
  __device__ __forceinline__ float l_total() const {
    float l = l_run + shfl_xor_f(l_run, 16);
    return l + shfl_xor_f(l, 32);
  }
};

// fp32 tile engine (pools, q and output in fp32) for RT 16-column row tiles, near the
// 16-bit engines' register layout, so the decode kernel around it -- the cross-wave
// combine, the split-K partials and their merge -- is the same:
//   S^T = K . Q^T on v_mfma_f32_16x16x4_f32: lane (g,n) loads dims 16c+4g .. +3
//     of key n and of column n's query (one 16-byte load per chunk c); MFMA
//     (c, j) contracts dim 16c + 4g + j in k-slot g.  -> lane (g,n) holds the
//     scores of column n for keys 4g..4g+3.
//   O^T += V^T . P^T, MFMA (w, j, r) taking keys 4g + r in k-slot g: A = V[key 4g+r]
//     [dim 64w + 4n + j] (one 16-byte load per (r, 64-dim group w); the 16 lanes of a
//     group read 256 consecutive bytes of a row), B = the lane's probability of key
//     4g + r.  -> lane (g,n) accumulates O[col n][64w + 4(4g + i) + j] in o[4w + j][i];
//     finish() turns each 4x4 of registers, so that o[x] then holds the 4 consecutive
//     dims from f32_dim0(x, g).
// Probabilities stay fp32; the online softmax is the 16-bit engines' (base 2,
// the same rescale slack).  Any block size: a table lookup per key row, or
// (LIST, block sizes that are multiples of 16) the wave's tile rows held one
// per lane.  Column n of row tile rt accepts keys < limit[rt] (decode: tok_end;
// prefill: its position + 1).
//
// What bounds it: 64 MFMAs of 32 cycles per 16-key tile and row tile at D = 128
// against 16 KB of loads.  The tile loads are raw buffer loads through one scalar
// descriptor per tile with loop-invariant lane offsets (rows past the extent read as
// zeros): 8 + 8 loads and no per-row addresses.  With a dword load per V element, 64-bit
// row addresses and a select per element the engine held 304 VGPRs, one wave per SIMD,
// and a tile took 3190 cycles; it now fits two (decode) or three (prefill) waves.
//
// PAD: the real head_dim dr is below D (a multiple of 4): rows are dr floats
// apart within a pool row, the dims past dr are zeros in K and V (not loaded,
// and not written by the page write), and q is zero there too.
__device__ __forceinline__ constexpr int f32_dim0(int x, int g) {
  return 64 * (x >> 2) + 16 * g + 4 * (x & 3);
}

template <int D, bool LIST = false, bool PAD = false, int RT = 1>
struct F32Core {
  static constexpr int NC = D / 16;  // 16-byte K and q chunks per lane
  static constexpr int NW = D / 64;  // 64-dim groups of V
  static constexpr int NX = D / 16;  // output tiles of 16 dims

  const float* k_pool;
  const float* v_pool;
  const int32_t* trow;  // block-table row of the sequence
  int64_t rs;           // elements per pool row (kv_heads * head_dim; LIST: 64 rs < 2^31)
  int hoff;             // kv_head * head_dim
  int dr;               // PAD: the real head_dim
  int W, NB, BS, bs_log2;
  int tok_end;          // keys >= tok_end are never read
  int limit[RT];        // this lane's column of each row tile accepts keys < limit
  float scale_log2;
  // optional fused page write of the decode token (position new_pos)
  const float* knew_row;
  const float* vnew_row;
  float* k_pool_w;
  float* v_pool_w;
  int new_pos;          // -1: none
  // the wave's tiles: t_first, t_first + step, ... (LIST: block sizes that are
  // multiples of 16, so a tile's 16 keys are consecutive rows of one block;
  // lane j of row_vec holds the pool row of the first key of tile list_base + j,
  // refilled every 64 tiles, so no table load sits between two tiles' loads)
  int t_first, step;
  int row_vec, list_base;

  f32x4 qv[RT][NC];
  float m_run[RT];
  float l_run[RT];
  f32x4 o[RT][NX];

  __device__ __forceinline__ int64_t pool_row(int tok) const {
    int page = tok >> bs_log2;
    page = page < W ? page : W - 1;
    const int blk = clamp_block(trow[page], NB);
    return (int64_t)blk * BS + (tok & (BS - 1));
  }
  // LIST: the pool rows of tiles k0 .. k0 + 63 of the wave's list
  __device__ __forceinline__ void fill_list(int k0) {
    list_base = k0;
    row_vec = (int)pool_row((t_first + (k0 + lane_id()) * step) * kTile);
  }
  // LIST: descriptor of tile k of a pool, from its first key's row to the end of its
  // last valid key's row (loads past it return zeros)
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const float* pool, int k,
                                                             int t0) const {
    const int64_t base = (int64_t)__builtin_amdgcn_readlane(row_vec, k - list_base) * rs + hoff;
    const uint64_t addr = reinterpret_cast<uint64_t>(pool + base);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)addr);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(addr >> 32));
    const int rows = tok_end - t0 < kTile ? tok_end - t0 : kTile;
    const int nrec = __builtin_amdgcn_readfirstlane(
        ((rows - 1) * (int)rs + (PAD ? dr : D)) * (int)sizeof(float));
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), 0,
                                             nrec, 0x00020000);
  }

  __device__ __forceinline__ void init_acc() {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      m_run[rt] = kNegInf;
      l_run[rt] = 0.f;
#pragma unroll
      for (int x = 0; x < NX; ++x) o[rt][x] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }

  // K of tile k: chunk c of key n.  Fills the tile list when tile k is past it, so it
  // runs before load_v of the same tile.
  __device__ __forceinline__ void load_k(int k, f32x4 (&kk)[NC]) {
    const int lane = lane_id();
    const int g = lane >> 4;
    const int n = lane & 15;
    const int t0 = (t_first + k * step) * kTile;
    if constexpr (LIST) {
      if (k - list_base >= kWave) fill_list(k);  // wave-uniform
      const __amdgpu_buffer_rsrc_t r = tile_rsrc(k_pool, k, t0);
      const uint32_t off = (uint32_t)((n * (int)rs + 4 * g) * (int)sizeof(float));
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if constexpr (PAD) kk[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!PAD || 16 * c + 4 * g < dr)
          kk[c] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 64 * c, 0, 0));
      }
    } else {
      const int tok = t0 + n < tok_end ? t0 + n : tok_end - 1;
      const float* row = k_pool + pool_row(tok) * rs + hoff + 4 * g;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        kk[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!PAD || 16 * c + 4 * g < dr) kk[c] = *reinterpret_cast<const f32x4*>(row + 16 * c);
      }
    }
    if (new_pos >= t0 && new_pos < t0 + kTile && t0 + n == new_pos) {
      float* row = k_pool_w + pool_row(new_pos) * rs + hoff + 4 * g;
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (!PAD || 16 * c + 4 * g < dr) {
          kk[c] = *reinterpret_cast<const f32x4*>(knew_row + 16 * c + 4 * g);
          *reinterpret_cast<f32x4*>(row + 16 * c) = kk[c];
        }
    }
  }

  // V of tile k: dims 64w + 4n .. +3 of key 4g + r (zeros for keys past tok_end).
  __device__ __forceinline__ void load_v(int k, f32x4 (&vv)[4][NW]) {
    const int lane = lane_id();
    const int g = lane >> 4;
    const int n = lane & 15;
    const int t0 = (t_first + k * step) * kTile;
    if constexpr (LIST) {
      // the row step is part of the lane offset: the range check that zeroes the keys past
      // tok_end is not promised to count a scalar offset
      const __amdgpu_buffer_rsrc_t b = tile_rsrc(v_pool, k, t0);
      const uint32_t off = (uint32_t)((4 * g * (int)rs + 4 * n) * (int)sizeof(float));
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          if constexpr (PAD) vv[r][w] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (!PAD || 64 * w + 4 * n < dr)
            vv[r][w] = __builtin_bit_cast(
                f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                           b, off + (uint32_t)(r * (int)rs * (int)sizeof(float)) + 256 * w, 0, 0));
        }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tv = t0 + 4 * g + r;
        const bool ok = tv < tok_end;
        const float* row = v_pool + pool_row(ok ? tv : tok_end - 1) * rs + hoff + 4 * n;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          f32x4 val = f32x4{0.f, 0.f, 0.f, 0.f};
          if (!PAD || 64 * w + 4 * n < dr) val = *reinterpret_cast<const f32x4*>(row + 64 * w);
          vv[r][w] = ok ? val : f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
    if (new_pos >= t0 && new_pos < t0 + kTile) {  // wave-uniform
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (t0 + 4 * g + r != new_pos) continue;
        float* row = v_pool_w + pool_row(new_pos) * rs + hoff + 4 * n;
#pragma unroll
        for (int w = 0; w < NW; ++w)
          if (!PAD || 64 * w + 4 * n < dr) {
            vv[r][w] = *reinterpret_cast<const f32x4*>(vnew_row + 64 * w + 4 * n);
            *reinterpret_cast<f32x4*>(row + 64 * w) = vv[r][w];
          }
      }
    }
  }

  // Scores of tile k's keys, then the online softmax: p[rt] = this lane's probabilities
  // (keys 4g .. 4g+3).  The dims are summed in two chains, so that no MFMA waits for
  // the one before it.
  __device__ __forceinline__ void scores(const f32x4 (&kk)[NC], f32x4 (&sacc)[RT]) const {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; c += 2)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          s0 = mfma4_f32(kk[c][j], qv[rt][c][j], s0);
          s1 = mfma4_f32(kk[c + 1][j], qv[rt][c + 1][j], s1);
        }
      sacc[rt] = s0 + s1;
    }
  }
  __device__ __forceinline__ void softmax(int k, const f32x4 (&sacc)[RT], f32x4 (&p)[RT]) {
    const int g = lane_id() >> 4;
    const int t0 = (t_first + k * step) * kTile;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float sv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        sv[i] = t0 + 4 * g + i < limit[rt] ? sacc[rt][i] * scale_log2 : kNegInf;
      float mx = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
      mx = fmaxf(mx, shfl_xor_f(mx, 16));
      mx = fmaxf(mx, shfl_xor_f(mx, 32));
      if (__ballot(mx > m_run[rt] + kRescaleSlack)) {  // wave-uniform
        const float m_new = fmaxf(m_run[rt], mx);
        const float alpha = m_new == kNegInf ? 1.f : exp2_fast(m_run[rt] - m_new);
        l_run[rt] *= alpha;
#pragma unroll
        for (int x = 0; x < NX; ++x) o[rt][x] *= alpha;
        m_run[rt] = m_new;
      }
      const float m_use = m_run[rt] == kNegInf ? 0.f : m_run[rt];
#pragma unroll
      for (int i = 0; i < 4; ++i) p[rt][i] = exp2_fast(sv[i] - m_use);
      l_run[rt] += (p[rt][0] + p[rt][1]) + (p[rt][2] + p[rt][3]);
    }
  }
  __device__ __forceinline__ void pv(const f32x4 (&vv)[4][NW], const f32x4 (&p)[RT]) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
            o[rt][4 * w + j] = mfma4_f32(vv[r][w][j], p[rt][r], o[rt][4 * w + j]);
  }
  __device__ __forceinline__ void compute_tile(int k, const f32x4 (&kk)[NC],
                                               const f32x4 (&vv)[4][NW]) {
    f32x4 sacc[RT], p[RT];
    scores(kk, sacc);
    softmax(k, sacc, p);
    pv(vv, p);
  }

  __device__ __forceinline__ int begin(int first, int stride, int t_end) {
    t_first = first;
    step = stride;
    const int ntiles = first < t_end ? (t_end - first + stride - 1) / stride : 0;
    if constexpr (LIST) {
      if (ntiles > 0) fill_list(0);
    }
    return ntiles;
  }

  // The wave's tiles t_first, t_first + step, ... below t_end, a whole tile of
  // prefetch (HBM-bound callers): while tile k is computed, the loads of tile k + 1
  // are in flight.
  __device__ __forceinline__ void run(int first, int stride, int t_end) {
    const int ntiles = begin(first, stride, t_end);
    if (ntiles == 0) return;
    f32x4 ka[NC], kb[NC];
    f32x4 va[4][NW], vb[4][NW];
    load_k(0, ka);
    load_v(0, va);
    for (int k = 0;; k += 2) {
      if (k + 1 < ntiles) {
        load_k(k + 1, kb);
        load_v(k + 1, vb);
      }
      compute_tile(k, ka, va);
      if (k + 1 >= ntiles) break;
      if (k + 2 < ntiles) {
        load_k(k + 2, ka);
        load_v(k + 2, va);
      }
      compute_tile(k + 1, kb, vb);
      if (k + 2 >= ntiles) break;
    }
    finish();
  }

  // The same with one register set (MFMA-bound callers, whose K/V come from the caches):
  // tile k + 1's K is loaded after tile k's scores and its V after tile k's products,
  // half a tile of MFMAs ahead of its use.  ntiles: begin()'s result, which the caller takes
  // ahead of its query loads: K waits for the table entries and then not for the queries too.
  __device__ __forceinline__ void run_single(int ntiles) {
    if (ntiles == 0) return;
    f32x4 kk[NC], vv[4][NW], sacc[RT], p[RT];
    load_k(0, kk);
    // K before V: with the two interleaved the loop waits for all of V ahead of the scores
    __builtin_amdgcn_sched_barrier(0);
    load_v(0, vv);
    for (int k = 0; k < ntiles; ++k) {
      scores(kk, sacc);
      if (k + 1 < ntiles) load_k(k + 1, kk);
      softmax(k, sacc, p);
      pv(vv, p);
      if (k + 1 < ntiles) load_v(k + 1, vv);
    }
    finish();
  }

  // Register transposes: o[rt][x] then holds 4 consecutive dims from f32_dim0(x, g).
  __device__ __forceinline__ void finish() {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        f32x4 t[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) t[i][j] = o[rt][4 * w + j][i];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[rt][4 * w + i] = t[i];
      }
  }

  __device__ __forceinline__ float l_total(int rt = 0) const {
    float l = l_run[rt] + shfl_xor_f(l_run[rt], 16);
    return l + shfl_xor_f(l, 32);
  }

  // After finish(): the four lanes of a row exchange 64-dim groups' chunks, so that o[x]
  // holds the 4 dims from 16x + 4g and one store of the four covers 64 consecutive bytes.
  __device__ __forceinline__ void to_row_order(f32x4 (&e)[NX]) const {
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t a[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = __float_as_uint(e[4 * w + i][j]);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const auto s = __builtin_amdgcn_permlane32_swap(a[i], a[i + 2], false, false);
          a[i] = s[0];
          a[i + 2] = s[1];
        }
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          const auto s = __builtin_amdgcn_permlane16_swap(a[i], a[i + 1], false, false);
          a[i] = s[0];
          a[i + 1] = s[1];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) e[4 * w + i][j] = __uint_as_float(a[i]);
      }
  }
};

// Fast path for block sizes that are multiples of 16: the 16 keys of a tile
// share one physical block, so a tile is fully described by wave-uniform
// values -- the pool row of its first key and its key count.  A wave's tiles
// form a list held one per lane (lane k: tile k, k < 64), filled from the block
// tables before the first load, so no table access sits between two tiles'
// K/V loads.
//
// PAD: the real head_dim is below D (D = the next of 64 / 128 / 256 computed):
// rows are nch 16-byte chunks long in the pool, the chunks past them are zeros
// in the K and V registers (q is zero there too) and never written.
template <int D, class E = Fp16, bool PAD = false>
struct TileListCore {
  using C = TileCfg<D>;

  const f16* k_pool;
  const f16* v_pool;
  int rs;                 // elements per pool row (kv_heads * head_dim)
  int hoff;               // kv_head * head_dim
  int nch;                // PAD: 16-byte chunks of a real row
  float scale_log2;
  unsigned char* stage;   // per-wave LDS tile, C::STAGE bytes
  int ntiles;             // tiles in the list (<= 64)
  int row_vec;            // lane k < ntiles: pool row (block * BS + offset) of tile k's first key
  int rows_vec;           // lane k < ntiles: keys in tile k (1..16)

  // The decoded token's K/V row (row new_row of tile new_tile; -1: not in this
  // list) comes from these registers instead of the pool, so no load waits on
  // the page write; the caller writes the row to the pool (store_new_row).
  int new_tile;
  int new_row;
  f16x8 knew[C::NK];      // lane (g, n): chunks 4s+g of the new K row
  f16x8 vnew;             // lane l: chunk l % CPR of the new V row

  f16x8 qv[C::NK];
  float m_run;
  float l_run;
  f32x4 o[C::NX];

  __device__ __forceinline__ void init_acc() {
    m_run = kNegInf;
    l_run = 0.f;
#pragma unroll
    for (int x = 0; x < C::NX; ++x) o[x] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // Element offset of row 0 of tile k (kv head included); wave-uniform.
  __device__ __forceinline__ int64_t tile_base(int k) const {
    return (int64_t)__builtin_amdgcn_readlane(row_vec, k & (kWave - 1)) * rs + hoff;
  }
  // Keys of tile k; 0 past the end of the list.
  __device__ __forceinline__ int tile_rows(int k) const {
    const int r = __builtin_amdgcn_readlane(rows_vec, k & (kWave - 1));
    return k < ntiles ? r : 0;
  }

  // Tile loads are raw buffer loads: a scalar descriptor per tile (base = row
  // 0 of the tile for this KV head, extent = the tile's keys) and a
  // loop-invariant 32-bit byte offset per lane.  Rows past the extent read as
  // zeros, so stale pool contents beyond a context never reach the
  // accumulators, and a tile past the list loads nothing.
  __device__ __forceinline__ uint32_t k_off0() const {
    const int lane = lane_id();
    return (uint32_t)(((lane & 15) * rs + (lane >> 4) * 8) * 2);
  }
  __device__ __forceinline__ static uint32_t k_soff(int s) { return (uint32_t)(s * 64); }
  __device__ __forceinline__ uint32_t v_off0() const {
    const int lane = lane_id();
    return (uint32_t)(((lane / C::CPR) * rs + (lane % C::CPR) * 8) * 2);
  }
  __device__ __forceinline__ uint32_t v_soff(int j) const { return (uint32_t)(j * C::RPI * rs * 2); }
  __device__ __forceinline__ static f16x8 buf_ld16(__amdgpu_buffer_rsrc_t r, uint32_t voff,
                                                   uint32_t soff) {
    return __builtin_bit_cast(f16x8,
                              __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, kPagePolicy));
  }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const f16* pool, int64_t base,
                                                             int rows) const {
    // Every field goes through readfirstlane: the values are wave-uniform, and
    // a descriptor held in vector registers would make the backend wrap each
    // load in a waterfall loop.
    const uint64_t addr = reinterpret_cast<uint64_t>(pool + base);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)addr);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(addr >> 32));
    // PAD: the extent ends at the real end of the last key's row, so the
    // chunks past it in that row read as zeros rather than past the pool
    const int nrec = __builtin_amdgcn_readfirstlane(
        PAD ? (rows > 0 ? ((rows - 1) * rs + nch * 8) * 2 : 0) : rows * rs * 2);
    void* p = reinterpret_cast<void*>(((uint64_t)hi << 32) | lo);
    // dword 3 = 0x00020000: 32-bit data format, the gfx9 setting for raw dword access
    return __builtin_amdgcn_make_buffer_rsrc(p, 0, nrec, 0x00020000);
  }

  // Issues the K/V loads of tile k; nothing here waits for data.
  __device__ __forceinline__ void load_tile(int k, f16x8 (&kk)[C::NK], f16x8 (&vv)[C::NK]) const {
    const int64_t base = tile_base(k);
    const int rows = tile_rows(k);
    const __amdgpu_buffer_rsrc_t kr = tile_rsrc(k_pool, base, rows);
    const __amdgpu_buffer_rsrc_t vr = tile_rsrc(v_pool, base, rows);
    const uint32_t ko = k_off0();
    const uint32_t vo = v_off0();
    if constexpr (PAD) {
      // only the real chunks of a row are loaded: the rest stay zeros
      const int lane = lane_id();
#pragma unroll
      for (int s = 0; s < C::NK; ++s) {
        kk[s] = f16x8{};
        if (4 * s + (lane >> 4) < nch) kk[s] = buf_ld16(kr, ko, k_soff(s));
      }
      const bool vin = lane % C::CPR < nch;
#pragma unroll
      for (int j = 0; j < C::NK; ++j) {
        vv[j] = f16x8{};
        if (vin) vv[j] = buf_ld16(vr, vo, v_soff(j));
      }
    } else {
#pragma unroll
      for (int s = 0; s < C::NK; ++s) kk[s] = buf_ld16(kr, ko, k_soff(s));
#pragma unroll
      for (int j = 0; j < C::NK; ++j) vv[j] = buf_ld16(vr, vo, v_soff(j));
    }
  }

  // One tile held in kk / vv: scores, V staging, softmax and PV.
  __device__ __forceinline__ void compute_tile(int k, f16x8 (&kk)[C::NK], f16x8 (&vv)[C::NK]) {
    const int lane = lane_id();
    const int vrow = lane / C::CPR;
    if (k == new_tile) {  // wave-uniform: substitute the decoded token's row
      const bool krow = (lane & 15) == new_row;
#pragma unroll
      for (int s = 0; s < C::NK; ++s) kk[s] = krow ? knew[s] : kk[s];
#pragma unroll
      for (int j = 0; j < C::NK; ++j) vv[j] = j * C::RPI + vrow == new_row ? vnew : vv[j];
    }
    f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < C::NK; ++s) {
      sacc = mma16<E>(lo4(kk[s]), lo4(qv[s]), sacc);
      sacc = mma16<E>(hi4(kk[s]), hi4(qv[s]), sacc);
    }
    compiler_fence();
    {
      const int cv = lane % C::CPR;
#pragma unroll
      for (int j = 0; j < C::NK; ++j) {
        const int r = j * C::RPI + vrow;
        unsigned char* dst = stage + r * C::ROWB + cv * 16;
        *reinterpret_cast<f16x8*>(dst) = vv[j];  // ROWB is a multiple of 16
      }
    }
    compiler_fence();
    softmax_pv_tile<D, E>(sacc, 0, tile_rows(k), scale_log2, stage, m_run, l_run, o);
    compiler_fence();
  }

  // Two register stages: while tile k is computed, the loads of tile k+1 are
  // in flight.  Loads are issued unconditionally (zero extent past the end of
  // the list), so the loop has no join points and every wait is exact.
  __device__ __forceinline__ void run() {
    f16x8 ka[C::NK], va[C::NK], kb[C::NK], vb[C::NK];
    load_tile(0, ka, va);
    for (int k = 0;; k += 2) {
      load_tile(k + 1, kb, vb);
      if (k >= ntiles) break;
      compute_tile(k, ka, va);
      load_tile(k + 2, ka, va);
      if (k + 1 >= ntiles) break;
      compute_tile(k + 1, kb, vb);
    }
  }

  // Writes the decoded token's K/V row to the pool (the wave holding its tile).
  __device__ __forceinline__ void store_new_row(f16* k_pool_w, f16* v_pool_w) const {
    if (new_tile < 0) return;
    const int lane = lane_id();
    const int64_t base = tile_base(new_tile);
    char* kb = reinterpret_cast<char*>(k_pool_w + base);
    char* vb = reinterpret_cast<char*>(v_pool_w + base);
    if ((lane & 15) == new_row) {
#pragma unroll
      for (int s = 0; s < C::NK; ++s)
        if (!PAD || 4 * s + (lane >> 4) < nch)
          *reinterpret_cast<f16x8*>(kb + k_off0() + k_soff(s)) = knew[s];
    }
    const int vrow = lane / C::CPR;
#pragma unroll
    for (int j = 0; j < C::NK; ++j)
      if (j * C::RPI + vrow == new_row && (!PAD || lane % C::CPR < nch))
        *reinterpret_cast<f16x8*>(vb + v_off0() + v_soff(j)) = vnew;
  }

  __device__ __forceinline__ float l_total() const {
    float l = l_run + shfl_xor_f(l_run, 16);
    return l + shfl_xor_f(l, 32);
  }
};

}  // namespace fe
