// Prefill GQA attention for gfx950: T new tokens per sequence attend causally
// to their sequence's cached keys (the prompt chunk's own K/V already
// appended by rope_append), over the reference's contiguous store or the
// paged pool, bf16 or fp8-e4m3 cache.
//
// Replaces the prefill branch of the reference's attention (attn.py:321-341:
// append, get_kv, then SDPA with is_causal=True at past_len 0 or the mask
// key_pos <= past_len + query_pos otherwise) for a ragged batch.
//
// One workgroup of 2, 4 or 8 waves (PrefillShape; which one: launch_d) per
// (sequence b, KV head hk, group of columns), a column being one (query token,
// head of the group) pair: a wave owns 32 of them (qt = 32 / G consecutive
// tokens) and walks the keys in tiles of 64 or 32 that the whole workgroup
// shares through LDS. Every thread loads its 16-byte
// pieces of the next tile's K and V into registers while the current tile is
// computed and writes them to the other LDS buffer afterwards (one barrier a
// tile); fp8 codes become bf16 on the way (exact), once per workgroup, so the
// compute loop is one for both cache types.
//
// Compute, per 32 keys and 32 columns, on v_mfma_f32_32x32x16_bf16:
//   S^T = K q^T   A = K rows from LDS (16-byte reads), B = q (registers)
//   softmax       a lane holds 16 keys of one column; the other 16 are in the
//                 lane 32 away, so only a moving maximum crosses lanes
//   O^T += V^T P^T  A = V read back transposed (ds_read_b64_tr_b16), B = P as
//                 bf16 P_hi + P_lo (~16 mantissa bits: a single bf16 P misses
//                 the 2e-3 absolute bound on short, cancelling rows). The order
//                 of the 16 contracted keys is the one S^T's layout leaves in
//                 each lane's registers, used for V as well: P needs no shuffle.
//
// Tiles below the workgroup's first token are whole for every column and run
// in a loop without masks; the others run in a loop of their own, in which a
// wave leaves out the 32 keys of Q K^T and the 16-key steps of P V past its last
// token and takes V past it as zero: the tile holds values of later waves'
// tokens, and an infinity or NaN there would reach this wave's columns as 0 x inf.
// Limit: within a wave that is what happens. An infinite or NaN value row turns
// the outputs of the earlier tokens that share its wave (32 / G of them, counted
// from the chunk's first) NaN in its head dim. Telling them apart takes a pass per
// key (20 to 57 registers spilled) or a check of each edge tile's V (short prompts
// 5-12 % slower); the fp32 kernel has it.
//
// Bound: the shared issue of VALU and matrix instructions. Per 32 x 32 block at
// D 64 a wave issues ~125 VALU instructions (16 exponentials; the P split is 48,
// the sums and the maxima 24) and 12 MFMAs; measured, 8 MFMAs and 64 FMAs of one
// SIMD take 200 ns where either alone takes 145-160, so the two overlap by
// half. With the same shape and timing-only loads of two fixed tiles the time
// does not move: K/V traffic does not bind. Against one wave per 64 columns
// streaming K/V for itself (K in registers, 16x16x32 MFMAs), calls on the same
// lengths drawn once (32 / 8 heads unless said):
//   64 x U[64, 2048]                             D 64   bf16  825 -> 725 us
//                                                       fp8   984 -> 797 us
//   4 x U[1024, 2048] after U[2048, 8192] cached D 128  fp8  1212 -> 896 us
//   8 x U[64, 4096]                              D 128  bf16  983 -> 777 us
//   1 x 20 after 8000 cached                     D 128  bf16  394 -> 226 us
//   6 x U[64, 2048], 32 / 4 heads                D 32   bf16   81 -> 67 us
// The last but one is bound otherwise: 8 workgroups, each walking its pair's 8020
// keys tile after tile, leave 248 CUs idle.
//
// With many pairs, all query blocks of one (sequence, KV head) run on one XCD,
// whose L2 keeps the pair's K/V for them (prefill_group).
#include <algorithm>
#include <type_traits>

#include "attn_tiles.h"
#include "tt_internal.h"
#include "tt_numerics.h"

namespace tt {
namespace {


typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x4t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Waves per workgroup (32 columns each), keys per LDS tile and the waves per SIMD
// that the registers must leave room for. bf16 at tile width <= 64 fits 128
// registers: two workgroups of 8 waves per CU. Width 128 (q and O alone take 96
// registers) runs one; fp8 at width 64 (the scales' registers) three of 4 waves.
// Wider workgroups read the pair's K/V from L2 less often; more waves per SIMD run
// one's softmax beside another's MFMAs. Measured (C5 prompts, D 64): 8 waves x
// two workgroups 717 us, two 32-column blocks a wave at two waves per SIMD 750,
// 4 waves x three 786; (prefix 2k-8k, fp8, D 128): 8 waves 1154-1190 us, 4
// waves x two 1171-1292, tiles of 128 keys 1289. Which shape runs: launch_d.
template <int kD, bool kIsFP8, int kWaves, int kTileKeys>
struct PrefillShape {
  static constexpr int D = kD;
  static constexpr bool kFP8 = kIsFP8;
  static constexpr int NW = kWaves;
  static constexpr int kOcc = D == 128 ? 2 : D == 64 && kFP8 ? 3 : 4;
  static constexpr int kKeys = kTileKeys;  // keys per LDS tile
  static constexpr int kThreads = 64 * NW;
  static constexpr int kRowBytes = 2 * D;           // LDS rows hold bf16
  static constexpr int kTileBytes = kKeys * kRowBytes;
  // LDS: K[2] | V[2] | fp8: K scales [2][kKeys], V scales [2][kKeys]
  static constexpr int kScaleAt = 4 * kTileBytes;
  static constexpr int kLds = kScaleAt + (kFP8 ? 4 * kKeys * 4 : 0);
};

// 16-byte chunk c of row r lies at chunk c ^ swizzle(r) of the row, so that
// 16 rows at one chunk (a K read's 16 lanes) resp. 4 rows of 64 bytes (a
// transposing V read's 32 lanes) fall on distinct banks.
template <int D>
__device__ __forceinline__ int k_swizzle(int r) {
  return D == 128 ? r & 15 : D == 64 ? (r >> 1) & 7 : (r >> 2) & 3;
}
template <int D>
__device__ __forceinline__ int v_swizzle(int r) {
  return D == 128 ? 4 * (r & 3) : D == 64 ? 4 * ((r >> 1) & 1) : 0;
}

// This thread's share of one tile on its way from the cache to LDS: N of the
// tile's 16-byte chunks, K's rows first, then V's.
template <class SH>
struct Staged {
  static constexpr int kChunks = SH::D * (SH::kFP8 ? 1 : 2) / 16;  // of a cached row
  static constexpr int kHalf = SH::kKeys * kChunks;        // K's chunks
  static constexpr int N = 2 * kHalf / SH::kThreads;
  static_assert(N * SH::kThreads == 2 * kHalf && kHalf % 64 == 0 && 64 / kChunks <= 16, "a wave: K or V, one block");
  u32x4 x[N];
  float scale[N];  // fp8: the row's scale, in the thread that holds the row's first chunk
  static __device__ __forceinline__ bool is_v(int j) {
    return __builtin_amdgcn_readfirstlane(threadIdx.x + j * SH::kThreads) >= kHalf;
  }
  static __device__ __forceinline__ int row(int j) {
    return (threadIdx.x + j * SH::kThreads) % kHalf / kChunks;
  }
  static __device__ __forceinline__ int chunk() { return threadIdx.x % kChunks; }
};

// Issue the loads of the tile at key t0. `entry` holds, one per lane, the
// page-table entries of pages pbase.. (see stream_block_addr); rows past L and
// chunks past a padded row's end read zero (the buffer range).
template <class SH, bool kPad>
__device__ __forceinline__ void stage_load(const DecodeArgs &a, int b, int hk, int L, int entry, int pbase, int t0,
                                           Staged<SH> &st) {
  using ST = Staged<SH>;
  constexpr int D = SH::D;
  constexpr bool kFP8 = SH::kFP8;
  constexpr int E = KVTraits<kFP8>::kElemBytes;
  const int hd = row_len<D, kPad>(a);
  const int c = ST::chunk();
#pragma unroll
  for (int j = 0; j < ST::N; ++j) {
    const int row = ST::row(j);
    const int blk = __builtin_amdgcn_readfirstlane(t0 / 16 + row / 16);
    int64_t elem;
    int rows;
    stream_block_addr<D, kPad>(a, b, hk, L, entry, pbase, blk, elem, rows);
    const char *base = static_cast<const char *>(ST::is_v(j) ? a.v_cache : a.k_cache) + elem * E;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(base), (short)0, rows * hd * E, kBufferFlags);
    const int off = (kPad && 16 * c >= hd * E) ? 0x7ffffff0 : (row & 15) * hd * E + 16 * c;
    st.x[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
    if constexpr (kFP8) {
      // the block starts a 16-row scale group (the host checks the strides)
      const float *sc = (ST::is_v(j) ? a.v_scale : a.k_scale) + fp8_scale_index(scale_row<D, kPad>(a, elem));
      const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(sc), (short)0, rows * 4, kBufferFlags);
      st.scale[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, c == 0 ? 4 * (row & 15) : 0x7ffffff0, 0, 0));
    }
  }
}

// The staged pieces into LDS buffer `buf` as bf16 rows.
template <class SH>
__device__ __forceinline__ void stage_store(const DecodeArgs &a, const Staged<SH> &st, char *lds, int buf) {
  using ST = Staged<SH>;
  constexpr int D = SH::D;
  constexpr bool kFP8 = SH::kFP8;
  const int c = ST::chunk();
#pragma unroll
  for (int j = 0; j < ST::N; ++j) {
    const int row = ST::row(j);
    const bool v = ST::is_v(j);  // uniform
    char *dst = lds + (buf + (v ? 2 : 0)) * SH::kTileBytes + row * SH::kRowBytes;
    const int f = v ? v_swizzle<D>(row) : k_swizzle<D>(row);
    if constexpr (kFP8) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *reinterpret_cast<bf16x8 *>(dst + 16 * ((2 * c + h) ^ f)) =
            fp8x8_to_bf16x8(u32x2{st.x[j][2 * h], st.x[j][2 * h + 1]});
      if (c == 0)  // K scales carry the softmax scale: scores come out in log2 units
        reinterpret_cast<float *>(lds + SH::kScaleAt)[(buf + (v ? 2 : 0)) * SH::kKeys + row] =
            v ? st.scale[j] : st.scale[j] * a.scale_log2;
    } else {
      *reinterpret_cast<u32x4 *>(dst + 16 * (c ^ f)) = st.x[j];
    }
  }
}

// Lazy running maximum: a column's reference moves only when a tile's maximum
// exceeds it by more than kLazyMax (log2 units), so P <= 2^kLazyMax (fp32 O and
// l and the bf16 P halves have the range) and most tiles need no rescale.
constexpr float kLazyMax = 7.0f;

// p (one lane's 8 softmax values of a contraction step) as bf16 P_hi + P_lo:
// P_lo = bf16(p - P_hi), the difference exact in fp32.
__device__ __forceinline__ void split_p(const float (&p)[8], bf16x8 &hi, bf16x8 &lo) {
  const f32x8 pv = {p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7]};
  hi = __builtin_convertvector(pv, bf16x8);
  f32x8 rem;
  const u32x4 hw = __builtin_bit_cast(u32x4, hi);  // P_hi back in fp32 from the packed halves
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    rem[2 * i] = p[2 * i] - __uint_as_float(hw[i] << 16);
    rem[2 * i + 1] = p[2 * i + 1] - __uint_as_float(hw[i] & 0xffff0000u);
  }
  lo = __builtin_convertvector(rem, bf16x8);
}

template <class SH, bool kPad>
__global__ __launch_bounds__(SH::kThreads, SH::kOcc) void prefill_attn_kernel(PrefillArgs a) {
  constexpr int D = SH::D;
  constexpr bool kFP8 = SH::kFP8;
  constexpr int kKeys = SH::kKeys;
  constexpr int NU = kKeys / 32;
  const auto mx2 = [](float u, float v) { return __builtin_elementwise_maximum(u, v); };
  const int hd = row_len<D, kPad>(a);
  __shared__ __attribute__((aligned(16))) char lds[SH::kLds];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5;
  const int n = lane & 31;

  int pair, grp;
  if (!prefill_group(a, pair, grp)) return;
  const int b = pair / a.hkv;
  const int hk = pair - b * a.hkv;
  const int nb = a.new_lens != nullptr ? min(max(a.new_lens[b], 0), a.num_new) : a.num_new;
  const int wg_tokens = a.qt * SH::NW;
  if (grp * wg_tokens >= nb) return;
  const int pos0 = a.positions[b];
  // keys of the workgroup resp. the wave: 0 .. its last token, never past the host's bound (the page table's reach)
  const int L = __builtin_amdgcn_readfirstlane(min(pos0 + min((grp + 1) * wg_tokens, nb), a.max_len));
  if (pos0 < 0 || L <= 0) return;
  const int t_first = grp * wg_tokens + wave * a.qt;
  const int t_end = min(t_first + a.qt, nb);
  const int Lw = t_first < nb ? __builtin_amdgcn_readfirstlane(min(pos0 + t_end, L)) : 0;
  // keys below the workgroup's first token's limit are whole for every column
  const int lim_min = __builtin_amdgcn_readfirstlane(min(pos0 + grp * wg_tokens + 1, L));

  const int G = a.group;
  const int tq = n / G;
  const int head = n - tq * G;
  const int tok = t_first + tq;
  const bool col_valid = tq < a.qt && tok < t_end;
  bf16x8 qf[D / 16];
  const uint16_t *q = static_cast<const uint16_t *>(a.q) + (int64_t)b * a.q_sb + (int64_t)(hk * G + head) * a.q_sh +
                      (int64_t)tok * a.q_st;
#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
    const int d = 16 * s + 8 * half;
    // loaded without a branch: from the tensor's first row where there is no value
    const bool in = col_valid && (!kPad || d < hd);
    u32x4 v = *reinterpret_cast<const u32x4 *>(in ? q + d : static_cast<const uint16_t *>(a.q));
    if (!in) v = u32x4{0u, 0u, 0u, 0u};
    qf[s] = __builtin_bit_cast(bf16x8, v);
  }
  f32x16 o[D / 32];
#pragma unroll
  for (int c = 0; c < D / 32; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[c][r] = 0.f;
  float m = kNegInf, l = 0.f;  // the column's reference maximum (log2 units); this lane's part of its sum

  // page-table entries of 64 pages (>= 16 tiles) at a time, one per lane
  const int tiles = (L + kKeys - 1) / kKeys;
  const int last_page = (L - 1) >> a.page_shift;
  int entry = 0, pbase = 0;
  auto fetch_entries = [&](int tile) {
    if (a.page_table != nullptr) {
      pbase = (kKeys * tile) >> a.page_shift;
      entry = a.page_table[(int64_t)b * a.max_pages + min(pbase + lane, last_page)];
    }
  };
  Staged<SH> st;
  fetch_entries(0);
  stage_load<SH, kPad>(a, b, hk, L, entry, pbase, 0, st);
  stage_store<SH>(a, st, lds, 0);
  __syncthreads();

  // this lane's K row and V rows (see k_swizzle / v_swizzle); XORed with the
  // chunk of a k step resp. a 32-column block
  const int ka0 = n * SH::kRowBytes + 16 * (half ^ k_swizzle<D>(n));
  const int vj = (lane >> 2) & 3, vq = lane & 3;  // key 4 half + vj, columns 4 vq .. + 3 of a 16-column group
  const int va0 = (4 * half + vj) * SH::kRowBytes +
                  16 * (v_swizzle<D>(4 * half + vj) + 2 * ((lane >> 4) & 1) + (vq >> 1)) + 8 * (vq & 1);
  // Between tiles one register holds both offsets (ka0 < 2^13, va0 < 2^12) and
  // the column's token in the wave (and the lane's half): with more, 128 registers do not do (a
  // reload in the loop would wait for the next tile's loads).
  const uint32_t packed = ka0 | (uint32_t)va0 << 13 | (uint32_t)(col_valid ? tq : 0) << 25 |
                          (uint32_t)half << 31;
  // One tile. A tile that some column may see only in part (kEdge) has code of its own:
  // branches between the P V steps keep one step's softmax from running beside another's
  // MFMAs (in every tile they cost 1-17 % of the kernel).
  auto step = [&](int i, auto edge_tile) {
    constexpr bool kEdge = decltype(edge_tile)::value;
    const bool more = i + 1 < tiles;
    if (more) {
      if ((kKeys * (i + 1)) % 1024 == 0) fetch_entries(i + 1);
      stage_load<SH, kPad>(a, b, hk, L, entry, pbase, kKeys * (i + 1), st);
    }
    __builtin_amdgcn_sched_barrier(0);
    const char *kb = lds + (i & 1) * SH::kTileBytes;
    const char *vb = kb + 2 * SH::kTileBytes;
    const float *sc = reinterpret_cast<const float *>(lds + SH::kScaleAt) + (i & 1) * kKeys;
    const int t0 = kKeys * i;
    if (t0 < Lw) {  // uniform
      uint32_t pk = packed;
      asm volatile("" : "+v"(pk));
      const int ka = pk & 0x1fff, va = (pk >> 13) & 0xfff;
      const int quad = 4 * (int)(pk >> 31);
      f32x16 S[NU];
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) S[u][r] = 0.f;
      if (NU == 1 || !kEdge || Lw - t0 > 32) {  // uniform
#pragma unroll
        for (int s = 0; s < D / 16; ++s)
#pragma unroll
          for (int u = 0; u < NU; ++u) {  // two independent chains
            const bf16x8 kf = *reinterpret_cast<const bf16x8 *>(kb + 32 * u * SH::kRowBytes + (ka ^ (32 * s)));
            S[u] = mfma32(kf, qf[s], S[u]);
          }
      } else {  // no token of the wave sees the second half
#pragma unroll
        for (int s = 0; s < D / 16; ++s)
          S[0] = mfma32(*reinterpret_cast<const bf16x8 *>(kb + (ka ^ (32 * s))), qf[s], S[0]);
      }
      if constexpr (kFP8) {  // K scales (times the softmax scale: log2 units)
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const f32x4 kc = *reinterpret_cast<const f32x4 *>(sc + 32 * u + 8 * x + quad);
#pragma unroll
            for (int r = 0; r < 4; ++r) S[u][4 * x + r] *= kc[r];
          }
      }
      if constexpr (kEdge) {
        const int lim = min(pos0 + t_first + (int)((pk >> 25) & 31) + 1, L);  // keys this column may see
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = t0 + 32 * u + 8 * (r >> 2) + (r & 3) + quad;
            S[u][r] = key < lim ? S[u][r] : kNegInf;
          }
      }
      float mx = S[0][0];  // nested pairs fold into three-input maxima
#pragma unroll
      for (int r = 1; r < 16 * NU - 1; r += 2) mx = mx2(mx2(mx, S[r >> 4][r & 15]), S[(r + 1) >> 4][(r + 1) & 15]);
      mx = mx2(mx, S[NU - 1][15]);
      // A column moves iff one of its two lanes' own maxima is past its
      // reference (always on the first tile: m = -inf, key 0 valid); only then
      // are they combined and O rescaled.
      if (__builtin_amdgcn_ballot_w64((kFP8 ? mx : mx * a.scale_log2) > m + kLazyMax) != 0) {  // uniform
        const auto p32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = mx2(__uint_as_float(p32[0]), __uint_as_float(p32[1]));
        if constexpr (!kFP8) mx *= a.scale_log2;
        const float m_new = mx > m + kLazyMax ? mx : m;
        const float alpha = __builtin_amdgcn_exp2f(m - m_new);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int c = 0; c < D / 32; ++c) o[c] *= alpha;
      }
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          if (kEdge && t0 + 32 * u + 16 * t >= Lw) continue;  // uniform: keys past the wave's last token
          bf16x8 vf[D / 32];
#pragma unroll
          for (int c = 0; c < D / 32; ++c) {
            bf16x4t part[2];
#pragma unroll
            for (int w = 0; w < 2; ++w)
              part[w] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4t *)(
                  vb + (32 * u + 16 * t + 8 * w) * SH::kRowBytes + (va ^ (64 * c))));
            vf[c] = bf16x8{part[0][0], part[0][1], part[0][2], part[0][3],
                           part[1][0], part[1][1], part[1][2], part[1][3]};
          }
          if (kEdge && t0 + 32 * u + 16 * t + 16 > Lw) {  // uniform: V past the wave's last token is zero
            const int left = Lw - (t0 + 32 * u + 16 * t + quad);
            u32x4 keep;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              const int r = 8 * (w >> 1) + 2 * (w & 1);
              keep[w] = (r < left ? 0xffffu : 0u) | (r + 1 < left ? 0xffff0000u : 0u);
            }
#pragma unroll
            for (int c = 0; c < D / 32; ++c)
              vf[c] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, vf[c]) & keep);
          }
          float p[8];
#pragma unroll
          for (int r = 0; r < 8; ++r)
            p[r] = __builtin_amdgcn_exp2f(kFP8 ? S[u][8 * t + r] - m
                                               : __builtin_fmaf(S[u][8 * t + r], a.scale_log2, -m));
          l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
          if constexpr (kFP8) {  // fold the V scales in; a row past the end has scale and P zero
#pragma unroll
            for (int x = 0; x < 2; ++x) {
              const f32x4 vc = *reinterpret_cast<const f32x4 *>(sc + 2 * kKeys + 32 * u + 16 * t + 8 * x + quad);
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const float pv = p[4 * x + r] * vc[r];
                p[4 * x + r] = kEdge && p[4 * x + r] == 0.f ? 0.f : pv;  // a masked token's scale may be infinite
              }
            }
          }
          bf16x8 hi, lo;
          split_p(p, hi, lo);
#pragma unroll
          for (int c = 0; c < D / 32; ++c) o[c] = mfma32(vf[c], lo, o[c]);  // the small terms first
#pragma unroll
          for (int c = 0; c < D / 32; ++c) o[c] = mfma32(vf[c], hi, o[c]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    // the other buffer's readers are done since the last barrier
    if (more) stage_store<SH>(a, st, lds, (i + 1) & 1);
    __syncthreads();
  };
  int i = 0;
  for (const int whole = min(lim_min / kKeys, tiles); i < whole; ++i) step(i, std::false_type{});
  for (; i < tiles; ++i) step(i, std::true_type{});

  // normalise and write: the lane's column, head_dim entries 32 c + 8 i + 4 half .. + 3
  const float sum = l + __shfl_xor(l, 32, 64);
  const float inv = sum > 0.f ? 1.0f / sum : 0.f;
  // the column again from the lane: its token and head would take registers through the loop
  int ln = lane;
  asm volatile("" : "+v"(ln));
  const int tq_out = (ln & 31) / G;
  const int tok_out = t_first + tq_out;
  if (tq_out >= a.qt || tok_out >= t_end) return;
  uint16_t *out = static_cast<uint16_t *>(a.out) + (int64_t)b * a.o_sb + (int64_t)tok_out * a.o_st +
                  (int64_t)(hk * G + (ln & 31) - tq_out * G) * a.o_sh;
#pragma unroll
  for (int c = 0; c < D / 32; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d0 = 32 * c + 8 * i + 4 * (ln >> 5);
      if (kPad && d0 >= hd) continue;  // columns past head_dim (hd is a multiple of 8)
      const uint2 w = make_uint2(pack_bf16x2(o[c][4 * i] * inv, o[c][4 * i + 1] * inv),
                                 pack_bf16x2(o[c][4 * i + 2] * inv, o[c][4 * i + 3] * inv));
      if (a.vec_out) {
        *reinterpret_cast<uint2 *>(out + d0) = w;
      } else {
        out[d0] = (uint16_t)w.x;
        out[d0 + 1] = (uint16_t)(w.x >> 16);
        out[d0 + 2] = (uint16_t)w.y;
        out[d0 + 3] = (uint16_t)(w.y >> 16);
      }
    }
}

template <class SH, bool kPad>
hipError_t launch_shape(PrefillArgs a, hipStream_t stream) {
  a.qt = 32 / a.group;  // group <= 16
  const int wg_tokens = a.qt * SH::NW;
  a.wg_per_pair = (a.num_new + wg_tokens - 1) / wg_tokens;
  return launch_prefill_groups(a, SH::kThreads, [&](dim3 grid, const PrefillArgs &args) {
    hipLaunchKernelGGL((prefill_attn_kernel<SH, kPad>), grid, dim3(SH::kThreads), 0, stream, args);
  });
}

// Which workgroup runs a call. Wide ones (64-key tiles; 8 waves, fp8 at width
// 64: 4) stage a pair's K/V once for many columns and hide its latency best, but
// they hold all their waves, LDS and registers also where a pair's columns fill
// few of the waves, and for a few keys one 64-key tile is a long chain. So with
// keys within one tile, or columns for at most 4 waves on more pairs than the GPU
// holds wide workgroups: 4 waves on 32-key tiles (at width 32 and columns for two
// waves, on twice as many pairs, 2 waves), of which a CU holds two to four times
// as many. fp8 at width 128, whose registers allow 8 waves a CU in any case:
//  * up to 4 waves of columns: a wave per pair streaming K/V for itself
//    (prefill_attn_stream.hip) for keys within one tile, and for one wave of
//    columns once two 4-wave workgroups a CU do not hold the pairs; 4 waves on
//    64-key tiles past a pair per CU; 8 waves below, whose staging is the fastest;
//  * more columns: 4 waves where that fills idle CUs or keys are few, 8 otherwise.
// Measured, us (G 4, T new tokens after P cached; pairs of (sequence, KV head)):
//             D   pairs     P    T   wide  chosen
//   bf16     32    2048     0    2   12.5     4.9   2 x 32
//   bf16     32    2048  1000    8   67.8    44.4   2 x 32
//   bf16     64     512     0    8    5.6     4.3   4 x 32
//   bf16     64    1024   250    8   21.4    15.8   4 x 32
//   bf16     64    1024  4000    8  194.0   194.3   4 x 32
//   bf16    128     256     0   64   16.7    13.8   4 x 32
//   bf16    128     512  1000    8   65.8    47.2   4 x 32
//   fp8      64    1024  1000    8   59.8    36.5   4 x 32
//   fp8     128       8     0   20    6.4     5.1   a wave each
//   fp8     128    1024  1000    8  140.7    56.5   a wave each
//   fp8     128     512  1000    8   69.8    46.4   4 x 64
//   fp8     128       8  4000  200  186.1   163.8   4 x 64
//   fp8     128     256     0  200   68.7    51.3   4 x 64
//   fp8     128     128  1000  200  127.0   (4 x 64: 136)  8 x 64
template <int D, bool kFP8, bool kPad>
hipError_t launch_d(const PrefillArgs &a, hipStream_t stream) {
  const int cus = device_cu_count();
  const int64_t pairs = (int64_t)a.batch * a.hkv;
  const int qt = 32 / a.group;                  // group <= 16
  const int waves = (a.num_new + qt - 1) / qt;  // that a pair's columns fill
  if constexpr (kFP8 && D == 128) {
    if (waves <= 4 && (a.max_len <= 64 || (waves == 1 && pairs > 2 * cus))) return launch_prefill_attn_stream_fp8(a, stream);
    const int64_t wg8 = pairs * ((waves + 7) / 8), wg4 = pairs * ((waves + 3) / 4);
    if (waves <= 4 ? pairs > cus : wg4 <= cus || (a.max_len <= 512 && wg8 > cus))
      return launch_shape<PrefillShape<D, kFP8, 4, 64>, kPad>(a, stream);
  } else {
    const int64_t slots = (int64_t)cus * (D == 128 ? 1 : kFP8 ? 3 : 2);  // wide workgroups that the GPU holds
    if constexpr (D == 32)
      if (waves <= 2 && pairs > 2 * slots) return launch_shape<PrefillShape<D, kFP8, 2, 32>, kPad>(a, stream);
    if (a.max_len <= 64 || (waves <= 4 && pairs > slots))
      return launch_shape<PrefillShape<D, kFP8, 4, 32>, kPad>(a, stream);
  }
  return launch_shape<PrefillShape<D, kFP8, kFP8 && D == 64 ? 4 : 8, 64>, kPad>(a, stream);
}

}  // namespace

hipError_t launch_prefill_attn(const PrefillArgs &a, CacheKind kind, int head_dim, hipStream_t stream) {
  const int D = tile_head_dim(head_dim, kind);
  const bool pad = D != head_dim;
  if (kind == CacheKind::kFP8) {
    if (D == 64) return pad ? launch_d<64, true, true>(a, stream) : launch_d<64, true, false>(a, stream);
    if (D == 128) return pad ? launch_d<128, true, true>(a, stream) : launch_d<128, true, false>(a, stream);
    return hipErrorInvalidValue;
  }
  if (D == 32) return pad ? launch_d<32, false, true>(a, stream) : launch_d<32, false, false>(a, stream);
  if (D == 64) return pad ? launch_d<64, false, true>(a, stream) : launch_d<64, false, false>(a, stream);
  if (D == 128) return pad ? launch_d<128, false, true>(a, stream) : launch_d<128, false, false>(a, stream);
  return hipErrorInvalidValue;
}

}  // namespace tt
