// Prefill GQA attention over an fp32 cache for gfx950: T new tokens per
// sequence attend causally to their sequence's cached keys (their own K/V
// already appended), fp32 throughout (the reference without autocast,
// attn.py:321-341, 420-423), over the contiguous store or the paged pool.
//
// One workgroup per (sequence, KV head, NB blocks of 16 columns), a column
// being one (query token, head of the group) pair; its four waves take the
// 32-key tiles in turn (wave w: tiles w, w + 4, ..), each with an online
// softmax of its own, and their states meet in LDS. Products run on
// v_mfma_f32_16x16x4_f32 (fp32 operands and accumulation). A lane's 16-byte
// loads are the operands as they are:
//   S^T = K q^T    lane (m + 16 g) reads K[key m][16 u + 4 g ..]: element i is
//                  k slot g of step (u, i); q is held in the same order
//   O^T += V^T P^T S^T leaves keys 4 g + r of column n in lane (n + 16 g), so
//                  step r contracts the keys {4 g + r}: lane (m + 16 g) reads
//                  V[key 4 g + r][64 j + 4 m ..], element c being row m of the
//                  output block with d = 64 j + 4 m + c. P needs no shuffle.
// K's registers are reloaded for the next tile once Q K^T has used them (the
// softmax and P V hide it), V's after P V. Tiles below the workgroup's first
// token's limit run in a loop without masks and without scratch accesses;
// the others in one of their own.
//
// Bound: in small batches the key walk of the longest column, a quarter of its
// tiles per wave one after the other (the fp32 matrix rate, 64 flop per cycle
// and SIMD, alone would allow a fifth of the time). Against one VALU workgroup
// per query row, which reads the whole K/V prefix per row (4 prompts of 579,
// 579, 828 and 226 tokens, 8 / 2 heads, D 64; 1.0 GFLOP): 1296 + 13 us (its
// merge) -> 42 us; 76 us while the scores and O lay in scratch memory.
#include <algorithm>
#include <type_traits>

#include "attn_tiles.h"
#include "tt_internal.h"

namespace tt {
namespace {

constexpr int kTile = 32;   // keys per tile: two 16-key blocks
constexpr int kWaves = 4;

template <int D>
struct BlockF32 {  // one 16-key block: K fragments by 16 head_dim entries, V fragments by contraction step
  f32x4 k[D / 16];
  f32x4 v[4][D <= 64 ? 1 : 2];
};

template <int D, bool kPad>
__device__ __forceinline__ auto block_rsrc(const PrefillArgs &a, const void *base, int64_t elem, int rows) {
  return __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char *>(static_cast<const char *>(base)) + elem * 4, (short)0, rows * row_len<D, kPad>(a) * 4,
      kBufferFlags);
}

// Rows past the sequence and entries past a padded row's head_dim (a multiple
// of 4) read zero through the buffer range.
template <int D, bool kPad>
__device__ __forceinline__ void load_k(const PrefillArgs &a, int64_t elem, int rows, int lane, BlockF32<D> &x) {
  const int hd = row_len<D, kPad>(a);
  const auto rs = block_rsrc<D, kPad>(a, a.k_cache, elem, rows);
#pragma unroll
  for (int u = 0; u < D / 16; ++u) {
    const int d = 16 * u + 4 * (lane >> 4);
    const int off = kPad && d >= hd ? 0x7ffffff0 : ((lane & 15) * hd + d) * 4;
    x.k[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
  }
}

template <int D, bool kPad>
__device__ __forceinline__ void load_v(const PrefillArgs &a, int64_t elem, int rows, int lane, BlockF32<D> &x) {
  const int hd = row_len<D, kPad>(a);
  const auto rs = block_rsrc<D, kPad>(a, a.v_cache, elem, rows);
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int j = 0; j < (D <= 64 ? 1 : 2); ++j) {
      const int d = 64 * j + 4 * (lane & 15);
      const int off = (D < 64 || kPad) && d >= hd ? 0x7ffffff0 : ((4 * (lane >> 4) + r) * hd + d) * 4;
      x.v[r][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
    }
}

template <int D>
__device__ __forceinline__ bool any_nonfinite(const BlockF32<D> (&x)[2]) {
  bool bad = false;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < (D <= 64 ? 1 : 2); ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) bad |= (__float_as_uint(x[h].v[r][j][i]) & 0x7f800000u) == 0x7f800000u;
  return __builtin_amdgcn_ballot_w64(bad) != 0;
}

// P V of one tile key by key, for a tile that some columns see only in part
// and whose V holds an infinity or NaN: a masked key's P is 0, and 0 times
// those would reach columns that do not attend to the key. Each step's product
// runs once per key slot, with the other three slots' V zero, and a column
// keeps it where it sees the key. Inlined, so that O and S stay in registers.
template <int D, int NB, int NO>
__device__ __forceinline__ void pv_masked(const BlockF32<D> (&x)[2], const f32x4 (&S)[NB][2], int t0, int lane,
                                          const int (&lim)[NB], f32x4 (&o)[NB][NO]) {
#pragma unroll 1
  for (int slot = 0; slot < 4; ++slot)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = t0 + 16 * h + 4 * slot + r;
#pragma unroll
        for (int c = 0; c < NO; ++c) {
          const float v = (lane >> 4) == slot ? x[h].v[r][c >> 2][c & 3] : 0.f;
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            const f32x4 sum = __builtin_amdgcn_mfma_f32_16x16x4f32(v, S[j][h][r], o[j][c], 0, 0, 0);
#pragma unroll
            for (int w = 0; w < 4; ++w) o[j][c][w] = key < lim[j] ? sum[w] : o[j][c][w];
          }
          __builtin_amdgcn_sched_barrier(0);  // one block's sums in registers at a time (width 128 has none to spare)
        }
      }
}

template <int D, bool kPad, int NB>
__global__ __launch_bounds__(64 * kWaves, 2) void prefill_f32_kernel(PrefillArgs a) {
  constexpr int NJ = D <= 64 ? 1 : 2;     // 64-entry groups of an output row
  constexpr int NO = 4 * NJ;              // output blocks
  constexpr int ROW = 64 * NJ + 4;        // LDS row of a column's output (padded)
  __shared__ float so[kWaves][16 * NB][ROW];
  __shared__ float sm[kWaves][16 * NB], sl[kWaves][16 * NB];
  const int hd = row_len<D, kPad>(a);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, g = lane >> 4;
  int pair, grp;
  if (!prefill_group(a, pair, grp)) return;
  const int b = pair / a.hkv;
  const int hk = pair - b * a.hkv;
  const int G = a.group;
  const int wg_tokens = a.qt * NB;
  const int t_first = grp * wg_tokens;
  const int nb = a.new_lens != nullptr ? min(max(a.new_lens[b], 0), a.num_new) : a.num_new;
  const int pos0 = a.positions[b];
  const int t_end = min(t_first + wg_tokens, nb);
  const int L = t_first < nb && pos0 >= 0 ? __builtin_amdgcn_readfirstlane(min(pos0 + t_end, a.max_len)) : 0;

  const int lim_min = min(pos0 + t_first + 1, L);  // tiles below it are whole for every column
  int lim[NB];
  float qf[NB][D / 4];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int tq = n / G;
    const int t = t_first + j * a.qt + tq;
    const bool valid = tq < a.qt && t < t_end;
    lim[j] = valid ? min(pos0 + t + 1, L) : 0;
    const float *q = static_cast<const float *>(a.q) + (int64_t)b * a.q_sb + (int64_t)(hk * G + n - tq * G) * a.q_sh +
                     (int64_t)t * a.q_st;
#pragma unroll
    for (int u = 0; u < D / 16; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 16 * u + 4 * g + i;
        qf[j][4 * u + i] = valid && (!kPad || d < hd) ? q[d] : 0.f;
      }
  }
  f32x4 o[NB][NO];
  float m[NB], l[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
#pragma unroll
    for (int c = 0; c < NO; ++c) o[j][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[j] = kNegInf;
    l[j] = 0.f;
  }

  // 64 page-table entries (at least 1024 tokens) at a time, one per lane
  constexpr int kSpan = 1024 / kTile;
  const int tiles = (L + kTile - 1) / kTile;
  for (int c0 = 0; c0 < tiles; c0 += kSpan) {
    const int c1 = min(tiles, c0 + kSpan);
    if (c0 + wave >= c1) break;  // uniform: this wave has no tile here or later
    int entry = 0, pbase = 0;
    if (a.page_table != nullptr) {
      pbase = (kTile * c0) >> a.page_shift;
      entry = a.page_table[(int64_t)b * a.max_pages + min(pbase + lane, (L - 1) >> a.page_shift)];
    }
    BlockF32<D> x[2];
    int64_t e[2];
    int rows[2];
    auto address = [&](int it) {
      stream_block_addr<D, kPad>(a, b, hk, L, entry, pbase, 2 * it, e[0], rows[0]);
      stream_block_addr<D, kPad>(a, b, hk, L, entry, pbase, 2 * it + 1, e[1], rows[1]);
    };
    address(c0 + wave);
#pragma unroll
    for (int h = 0; h < 2; ++h) load_k<D, kPad>(a, e[h], rows[h], lane, x[h]);
#pragma unroll
    for (int h = 0; h < 2; ++h) load_v<D, kPad>(a, e[h], rows[h], lane, x[h]);
    // One tile. A tile that some column may see only in part (kEdge) has code of its own: the masks and the
    // registers of the key-by-key path stay out of the others'.
    auto step = [&](int it, auto edge_tile) {
      constexpr bool kEdge = decltype(edge_tile)::value;
      f32x4 S[NB][2];
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) S[j][h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < D / 16; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < NB; ++j)
              S[j][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[h].k[u][i], qf[j][4 * u + i], S[j][h], 0, 0, 0);
      address(min(it + kWaves, c1 - 1));  // past the span: loaded again, unused
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; ++h) load_k<D, kPad>(a, e[h], rows[h], lane, x[h]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        float mx = kNegInf;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = kTile * it + 16 * h + 4 * g + r;
            S[j][h][r] = !kEdge || key < lim[j] ? S[j][h][r] * a.scale_log2 : kNegInf;
            mx = fmaxf(mx, S[j][h][r]);
          }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m[j], mx);
        const float ref = m_new == kNegInf ? 0.f : m_new;  // no key of this column yet
        const float alpha = __builtin_amdgcn_exp2f(m[j] - ref);
        m[j] = m_new;
        float sum = 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            S[j][h][r] = __builtin_amdgcn_exp2f(S[j][h][r] - ref);
            sum += S[j][h][r];
          }
        l[j] = l[j] * alpha + sum;
#pragma unroll
        for (int c = 0; c < NO; ++c) o[j][c] *= alpha;
      }
      if (kEdge && any_nonfinite<D>(x)) {  // uniform; see pv_masked
        pv_masked<D, NB, NO>(x, S, kTile * it, lane, lim, o);
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < NO; ++c)
#pragma unroll
              for (int j = 0; j < NB; ++j)
                o[j][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[h].v[r][c >> 2][c & 3], S[j][h][r], o[j][c], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; ++h) load_v<D, kPad>(a, e[h], rows[h], lane, x[h]);
      __builtin_amdgcn_sched_barrier(0);
    };
    int it = c0 + wave;
    for (const int whole = min(lim_min / kTile, c1); it < whole; it += kWaves) step(it, std::false_type{});
    for (; it < c1; it += kWaves) step(it, std::true_type{});
  }

#pragma unroll
  for (int j = 0; j < NB; ++j) {
    float sum = l[j];
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (g == 0) {
      sm[wave][16 * j + n] = m[j];
      sl[wave][16 * j + n] = sum;
    }
    // block c = 4 j2 + e, row 4 g + r: d = 64 j2 + 4 (4 g + r) + e
#pragma unroll
    for (int c = 0; c < NO; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) so[wave][16 * j + n][64 * (c >> 2) + 4 * (4 * g + r) + (c & 3)] = o[j][c][r];
  }
  __syncthreads();
  // rows t >= new_lens[b] are written as zeros
  const int t_stop = min(t_first + wg_tokens, a.num_new);
  for (int i = threadIdx.x; i < 16 * NB * 64 * NJ; i += 64 * kWaves) {
    const int col = i / (64 * NJ), d = i % (64 * NJ);
    const int tq = (col & 15) / G;
    const int t = t_first + (col >> 4) * a.qt + tq;
    if (d >= hd || tq >= a.qt || t >= t_stop) continue;
    float v = 0.f;
    if (t < nb && L > 0) {
      float top = sm[0][col];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) top = fmaxf(top, sm[w][col]);  // finite: key 0 is every token's
      float num = 0.f, den = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float f = __builtin_amdgcn_exp2f(sm[w][col] - top);
        num += f * so[w][col][d];
        den += f * sl[w][col];
      }
      v = num / den;
    }
    static_cast<float *>(a.out)[(int64_t)b * a.o_sb + (int64_t)t * a.o_st +
                                (int64_t)(hk * G + (col & 15) - tq * G) * a.o_sh + d] = v;
  }
}

template <int D, bool kPad, int NB>
hipError_t launch_nb(PrefillArgs a, hipStream_t stream) {
  a.qt = 16 / a.group;  // group <= 16
  const int wg_tokens = a.qt * NB;
  a.wg_per_pair = (a.num_new + wg_tokens - 1) / wg_tokens;
  return launch_prefill_groups(a, 64 * kWaves, [&](dim3 grid, const PrefillArgs &args) {
    hipLaunchKernelGGL((prefill_f32_kernel<D, kPad, NB>), grid, dim3(64 * kWaves), 0, stream, args);
  });
}

// Two column blocks per workgroup halve the K/V reads per product; one spreads
// a small batch over more CUs. Two blocks from two workgroups per CU on
// (head_dim 128: its registers allow one).
template <int D, bool kPad>
hipError_t launch_d(const PrefillArgs &a, hipStream_t stream) {
  if constexpr (D <= 64) {
    const int64_t wgs = (int64_t)a.batch * a.hkv * ((a.num_new + 32 / a.group - 1) / (32 / a.group));
    if (wgs >= 2 * (int64_t)device_cu_count()) return launch_nb<D, kPad, 2>(a, stream);
  }
  return launch_nb<D, kPad, 1>(a, stream);
}

}  // namespace

bool prefill_f32_supported(int64_t head_dim) { return head_dim > 0 && head_dim <= 128 && head_dim % 4 == 0; }

hipError_t launch_prefill_attn_f32(const PrefillArgs &a, int head_dim, hipStream_t stream) {
  if (head_dim <= 32) return head_dim == 32 ? launch_d<32, false>(a, stream) : launch_d<32, true>(a, stream);
  if (head_dim <= 64) return head_dim == 64 ? launch_d<64, false>(a, stream) : launch_d<64, true>(a, stream);
  return head_dim == 128 ? launch_d<128, false>(a, stream) : launch_d<128, true>(a, stream);
}

}  // namespace tt
