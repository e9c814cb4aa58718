// Prefill GQA attention for gfx950, a wave per 32 (token, head) columns of a
// (sequence, KV head) pair: fp8 caches at tile width 128 with few new tokens, for
// keys within one tile, or where a pair's columns fill one wave and there are more
// pairs than the GPU holds of prefill_attn.hip's workgroups (a speculated or
// streamed turn of a full batch). Those share converted K/V tiles among waves,
// which here would have no columns, and hold 66 KB of LDS for it.
//
// A wave streams K/V for itself as the decode kernel does: K of the next
// 32-token tile in registers, V through its own 8 KB of LDS, both as fp8, on
// 16x16x32 MFMAs; two blocks of 16 columns use every tile. Keys past the wave's
// last token are not read; within the wave an infinite or NaN value row reaches
// earlier tokens, as in prefill_attn.hip.
//
// Bound: the cache's bytes. 1024 pairs, 2 tokens after 2000, head_dim 128
// (524 MB): 105-108 us; 8-wave workgroups sharing K/V 264 us (a round of 256
// pairs each), 2 waves on 32-key tiles 127 us.
#include "attn_tiles.h"
#include "tt_internal.h"
#include "tt_numerics.h"

namespace tt {
namespace {

constexpr int kD = 128;
constexpr int kNDB = kD / 32;
constexpr int kBlocks = 2;      // 16-column blocks a wave
constexpr int kSpanTiles = 16;  // tiles per page-table fetch (64 pages of at least 16 tokens cover them) and pipelined run

template <bool kPad>
__global__ __launch_bounds__(64, 2) void prefill_stream_kernel(PrefillArgs a) {
  using TR = KVTraits<true>;
  constexpr int NU = Tile<kD, true>::NU;
  constexpr int kKLoads = 2 * NU + 4;  // a tile's K fragments and scales
  __shared__ __attribute__((aligned(16))) char vlds[Tile<kD, true>::kVBytes];
  const int hd = row_len<kD, kPad>(a);
  const int lane = threadIdx.x;
  // rows past the sequence are not written by the V loads: they hold zeros or an earlier tile's values
  for (int i = lane; i < Tile<kD, true>::kVBytes / 16; i += 64) reinterpret_cast<u32x4 *>(vlds)[i] = u32x4{0u, 0u, 0u, 0u};
  __syncthreads();  // before any load to LDS

  int pair, grp;
  if (!prefill_group(a, pair, grp)) return;
  const int b = pair / a.hkv;
  const int hk = pair - b * a.hkv;
  const int nb = a.new_lens != nullptr ? min(max(a.new_lens[b], 0), a.num_new) : a.num_new;
  const int t_first = grp * a.qt * kBlocks;
  if (t_first >= nb) return;
  const int pos0 = a.positions[b];
  const int t_end = min(t_first + a.qt * kBlocks, nb);
  // keys the wave needs: 0 .. its last token, never past the host's bound (the page table's reach)
  const int L = __builtin_amdgcn_readfirstlane(min(pos0 + t_end, a.max_len));
  if (pos0 < 0 || L <= 0) return;

  const int G = a.group;
  const int n = lane & 15;
  const int g = lane >> 4;
  const int tq = n / G;
  const int head = n - tq * G;
  int lim[kBlocks];  // keys each block's column may see (a column without a token: key 0, with q zero)
  bf16x8 qf[kBlocks][kNDB];
  const uint16_t *q = static_cast<const uint16_t *>(a.q);
#pragma unroll
  for (int j = 0; j < kBlocks; ++j) {
    const int t = t_first + j * a.qt + tq;
    const bool valid = tq < a.qt && t < t_end;
    lim[j] = valid ? min(pos0 + t + 1, L) : 1;
    const int64_t row = (int64_t)b * a.q_sb + (int64_t)(hk * G + head) * a.q_sh + (int64_t)t * a.q_st;
#pragma unroll
    for (int s = 0; s < kNDB; ++s) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (valid && (!kPad || TR::q_offset(s, g) < hd)) v = *reinterpret_cast<const u32x4 *>(q + row + TR::q_offset(s, g));
      qf[j][s] = __builtin_bit_cast(bf16x8, v);
    }
  }
  bf16x8 ident16[2];
  u32x2 ident8[2];
  make_identity(lane, ident16, ident8);
  WaveState<kD, true> st[kBlocks];
#pragma unroll
  for (int j = 0; j < kBlocks; ++j) {
#pragma unroll
    for (int c = 0; c < 2 * kNDB; ++c) st[j].o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    st[j].m = kNegInf;
    st[j].l = 0.f;
  }

  // The decode kernel's pipeline: K(k + 1) | Q K^T, softmax | wait for V(k), read it | V(k + 1) | P V,
  // with explicit vmcnt counts (loads return in issue order). Every tile issues the next one's loads, the
  // last of a span its own again: the counts, and no branch round the loads (with one, 143 us for 105 above).
  const int tiles = (L + kTileTokens - 1) / kTileTokens;
  for (int c0 = 0; c0 < tiles; c0 += kSpanTiles) {
    const int c1 = min(tiles, c0 + kSpanTiles);
    int entry = 0, pbase = 0;
    if (a.page_table != nullptr) {
      pbase = (kTileTokens * c0) >> a.page_shift;
      entry = a.page_table[(int64_t)b * a.max_pages + min(pbase + lane, (L - 1) >> a.page_shift)];
    }
    Tile<kD, true> buf[2];
    int64_t e[2];
    int rows[2];
    auto load_k = [&](int it, Tile<kD, true> &x) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        stream_block_addr<kD, kPad>(a, b, hk, L, entry, pbase, 2 * it + h, e[h], rows[h]);
        load_k_block<kD, true, kPad>(a, e[h], rows[h], lane, x.k[h], x.ks[h], x.vs[h]);
      }
    };
    auto load_v = [&]() {
#pragma unroll
      for (int h = 0; h < 2; ++h) load_v_block_lds<kD, true, kPad>(a, e[h], rows[h], lane, vlds + h * NU * 1024);
    };
    auto tile = [&](int it, const Tile<kD, true> &cur, Tile<kD, true> &next) {
      int ahead = min(it + 1, c1 - 1);
      asm volatile("" : "+s"(ahead));  // loads of its own for the compiler also where it repeats the tile
      load_k(ahead, next);
      __builtin_amdgcn_sched_barrier(0);
      bf16x8 hi[kBlocks], lo[kBlocks];
#pragma unroll
      for (int j = 0; j < kBlocks; ++j)
        qk_softmax<kD, true>(a.scale_log2, kTileTokens * it, lim[j], lane, cur, qf[j], st[j], hi[j], lo[j]);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(vmcnt_only(kKLoads));  // this tile's V is in LDS
      VRegs<kD, true> vr;
      read_v<kD, true>(vlds, lane, vr);
      __builtin_amdgcn_s_waitcnt(kLgkmcntZero);
      __builtin_amdgcn_sched_barrier(0);
      load_v();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 2 * kNDB; ++c) {
        const bf16x8 vb = v_block<kD, true>(vr, c, ident8);
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) {
          st[j].o[c] = mfma_bf16(vb, lo[j], st[j].o[c]);  // the small terms first
          st[j].o[c] = mfma_bf16(vb, hi[j], st[j].o[c]);
        }
      }
    };
    load_k(c0, buf[0]);
    __builtin_amdgcn_sched_barrier(0);
    load_v();
    __builtin_amdgcn_sched_barrier(0);
    int it = c0;
    for (; it + 1 < c1; it += 2) {
      tile(it, buf[0], buf[1]);
      tile(it + 1, buf[1], buf[0]);
    }
    if (it < c1) {
      tile(it, buf[0], buf[1]);
      // without a reader the compiler drops the prefetch, and the count above would wait for too little
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int u = 0; u < NU; ++u) asm volatile("" ::"v"(buf[1].k[h][u]));
        asm volatile("" ::"v"(buf[1].ks[h]), "v"(buf[1].vs[h]));
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
  }

  // normalise and write: lane (n + 16 g) holds column n's entries o_col_d(c, 4 g) .. + 3 of every block c
  uint16_t *out = static_cast<uint16_t *>(a.out);
#pragma unroll
  for (int j = 0; j < kBlocks; ++j) {
    const int t = t_first + j * a.qt + tq;
    float l = st[j].l;
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    if (tq >= a.qt || t >= t_end) continue;
    const int64_t row = (int64_t)b * a.o_sb + (int64_t)t * a.o_st + (int64_t)(hk * G + head) * a.o_sh;
#pragma unroll
    for (int c = 0; c < 2 * kNDB; ++c) {
      const int d0 = o_col_d<true>(c, 4 * g);
      if (kPad && d0 >= hd) continue;  // columns past head_dim (a multiple of 16)
      const uint2 w = make_uint2(pack_bf16x2(st[j].o[c][0] * inv, st[j].o[c][1] * inv),
                                 pack_bf16x2(st[j].o[c][2] * inv, st[j].o[c][3] * inv));
      if (a.vec_out) {
        *reinterpret_cast<uint2 *>(out + row + d0) = w;
      } else {
        out[row + d0] = (uint16_t)w.x;
        out[row + d0 + 1] = (uint16_t)(w.x >> 16);
        out[row + d0 + 2] = (uint16_t)w.y;
        out[row + d0 + 3] = (uint16_t)(w.y >> 16);
      }
    }
  }
}

}  // namespace

hipError_t launch_prefill_attn_stream_fp8(PrefillArgs a, hipStream_t stream) {
  a.qt = 16 / a.group;  // group <= 16
  const int wave_tokens = a.qt * kBlocks;
  a.wg_per_pair = (a.num_new + wave_tokens - 1) / wave_tokens;
  return launch_prefill_groups(a, 64, [&](dim3 grid, const PrefillArgs &args) {
    if (a.head_dim == kD)
      hipLaunchKernelGGL((prefill_stream_kernel<false>), grid, dim3(64), 0, stream, args);
    else
      hipLaunchKernelGGL((prefill_stream_kernel<true>), grid, dim3(64), 0, stream, args);
  });
}

}  // namespace tt
