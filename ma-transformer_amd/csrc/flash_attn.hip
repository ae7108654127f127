// flash_attn.hip -- launches of the banded MFMA kernels (flash_kernel.h).
#include "flash_attn.h"

#include <algorithm>
#include <cmath>

#include "flash_kernel.h"
#include "host_common.h"

namespace ma_flash {

using namespace ma_dev;

namespace {

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
int64_t elt_of(const ma_attn_desc* d) { return d->dtype == MA_ATTN_F32 ? 4 : 2; }

// The band a descriptor maps to, clipped to the sequence.
struct Band {
  int64_t left, right, dil, nr;
};
bool band_of(const ma_attn_desc* d, Band* b) {
  if (d->pattern == MA_ATTN_DENSE) {
    *b = Band{d->seq_len, d->causal ? 0 : d->seq_len, 1, d->seq_len};
    return true;
  }
  if (d->pattern != MA_ATTN_SLIDING || d->left < 0 || d->right < 0) return false;
  const int64_t dil = std::min(d->dilation, std::max<int64_t>(d->seq_len, 1));  // classes past the rows are empty
  const int64_t nr = (d->seq_len + dil - 1) / dil;
  *b = Band{std::min(d->left, nr), std::min(d->right, nr), dil, nr};
  return true;
}

FlArgs args_of(const ma_attn_desc* d) {
  Band b;
  band_of(d, &b);
  FlArgs a{};
  a.N = d->seq_len;
  a.H = (int32_t)d->num_heads;
  a.D = (int32_t)d->head_dim;
  a.left = (int32_t)b.left;
  a.right = (int32_t)b.right;
  a.dil = (int32_t)b.dil;
  a.tok_bytes = (uint32_t)(b.dil * d->num_heads * d->head_dim * elt_of(d));
  a.scale = d->scale > 0.0f ? d->scale : 1.0f / std::sqrt(static_cast<float>(d->head_dim));
  a.scale_log2 = a.scale * 1.4426950408889634f;
  // rows that see more of the sequence the later they are run first
  a.desc = b.left >= b.nr && b.right < b.nr;
  return a;
}

template <typename T, int ND, int NQ, int NW, int KB, int OCC, int NPB = FlElt<T>::NPB, bool GL = false>
int run_fwd(const ma_attn_desc* d, FlArgs a, hipStream_t st) {
  Band b;
  band_of(d, &b);
  constexpr int QT = 16 * NQ * NW;
  constexpr size_t shm = 2 * FlStage<T, ND, KB, NW>::kMat;
  auto kern = &flash_fwd_kernel<T, ND, NQ, NW, KB, NPB, OCC, GL>;
  if (ma_host::reserve_lds(reinterpret_cast<const void*>(kern), shm, st)) return 1;
  a.tiles = (int32_t)((b.nr + QT - 1) / QT);
  const int64_t wgs = d->batch * d->num_heads * b.dil * a.tiles;
  ma_host::launch(true, kern, dim3((unsigned)wgs), dim3(64 * NW), (uint32_t)shm, st, a);
  return 0;
}

// Causal rows, the longest and the shortest tile of a stream in one workgroup.
template <typename T, int ND, int NW, int KB>
int run_pair(const ma_attn_desc* d, FlArgs a, hipStream_t st) {
  Band b;
  band_of(d, &b);
  constexpr int QT = 16 * NW;
  constexpr size_t shm = 2 * FlStage<T, ND, KB, NW>::kMat;
  auto kern = &flash_pair_fwd_kernel<T, ND, 1, NW, KB, FlElt<T>::NPB>;
  if (ma_host::reserve_lds(reinterpret_cast<const void*>(kern), shm, st)) return 1;
  a.desc = 0;
  a.tiles = (int32_t)((b.nr + QT - 1) / QT);
  const int64_t wgs = d->batch * d->num_heads * b.dil * a.tiles;
  ma_host::launch(true, kern, dim3((unsigned)wgs), dim3(64 * NW), (uint32_t)shm, st, a);
  return 0;
}

// One query group per wave, 4 waves, 64-key blocks in one buffer: measured
// best of 1 or 2 groups, 4 or 8 waves, 32- or 64-key blocks and one or two
// buffers at head_dim 32 and 128, in a first version (causal 128-key window, bf16,
// head_dim 128, 8 heads, 32768 rows: 83 us against 87-104, 75 now; two-sided
// 64-key window, head_dim 32, 4 x 8 heads, 8191 rows: f16 26 us against 28-31, f32
// 43 us against 43-70, 39 now).  16-bit windows of at most 128 keys at head_dim 32
// take 128-key blocks: a 64-query tile of a 64-key window is then one block (22 us
// against 24 on the f16 window above, 19.5 now).  float32 above head_dim 64 takes 32-key blocks
// (three planes of 64 rows would leave one workgroup per CU, or spill).
//
// Causal rows whose 128-row tiles are at most one per CU run in pairs, longest
// with shortest (float32, head_dim 64, 8 heads of 4000 rows: 136 us against
// 173 unpaired; above one tile per CU the scheduler evens the tiles out: 8000
// rows 415 us unpaired, 442 paired), past two 64-row tiles (float32, head_dim 64,
// 100 rows: 8.4 us, paired 10.1); not the 16-bit windows at head_dim 64 ([i-300,
// i] on 200 rows: 6.4 us, paired 9.3).
//
// float32 at head_dim 33 to 64 splits every staged row into three planes, so 8
// waves share a block once there are workgroups enough for every CU (two-sided
// 129-key window, 8 heads of 32768 rows: 82 us against 102 with 4 waves; 2
// heads of 600 rows: 14.7 against 11.8), and two query groups per wave pay on
// very long dense rows (causal, 8 heads of 16384 rows: 1275 us against 1387; 8000
// rows: 558 against 415).  Sequences of one 64-row tile would leave half of the 8
// waves idle.
template <typename T, int ND>
int fwd_nd(const ma_attn_desc* d, const FlArgs& a, hipStream_t st) {
  constexpr bool f32 = sizeof(T) == 4;
  constexpr int KB = f32 && ND > 2 ? 32 : 64;
  Band b;
  band_of(d, &b);
  const int64_t tiles128 = d->batch * d->num_heads * b.dil * ((b.nr + 127) / 128);
  if (a.desc && b.nr > 128 && tiles128 <= 256 && (f32 || d->head_dim != 64)) return run_pair<T, ND, 8, KB>(d, a, st);
  if constexpr (f32 && ND == 2) {
    if (d->pattern == MA_ATTN_DENSE && tiles128 >= 1024) return run_fwd<T, ND, 2, 8, KB, 2>(d, a, st);
    if (b.nr > 64 && tiles128 >= 256) return run_fwd<T, ND, 1, 8, KB, 2>(d, a, st);
  }
  // head_dim 64 in 16 bits: P in 16 bits, as in the stream kernel that these
  // windows took before; four workgroups to a CU
  if constexpr (!f32 && ND == 2)
    if (d->head_dim == 64) return run_fwd<T, ND, 1, 4, KB, 4, 1>(d, a, st);
  if constexpr (!f32 && ND == 1)
    if (b.left + b.right < 128) return run_fwd<T, ND, 1, 4, 128, 3>(d, a, st);
  return run_fwd<T, ND, 1, 4, KB, f32 ? 2 : 3>(d, a, st);
}

template <typename T>
int fwd_t(const ma_attn_desc* d, const FlArgs& a, hipStream_t st) {
  switch ((d->head_dim + 31) / 32) {
    case 1: return fwd_nd<T, 1>(d, a, st);
    case 2: return fwd_nd<T, 2>(d, a, st);
    case 3: return fwd_nd<T, 3>(d, a, st);
    default: return fwd_nd<T, 4>(d, a, st);
  }
}

template <typename T, int ND, int NQ, int NK, int NWQ, int NWK, int KB, int NPB, int OCC, bool SAVED, bool FAST, bool PAIR>
int run_bwd(const ma_attn_desc* d, FlArgs a, hipStream_t st) {
  Band b;
  band_of(d, &b);
  constexpr int QT = 16 * NQ * NWQ, KT = 16 * NK * NWK;
  constexpr size_t shm_q = 2 * FlStage<T, ND, KB, NWQ>::kMat;
  constexpr size_t shm_k = 2 * FlStage<T, ND, KB, NWK>::kMat + 2 * KB * sizeof(float);
  auto kq = &flash_dq_kernel<T, ND, NQ, NWQ, KB, NPB, OCC, SAVED, FAST, PAIR>;
  auto kk = &flash_dkv_kernel<T, ND, NK, NWK, KB, NPB, OCC, FAST, PAIR>;
  if (ma_host::reserve_lds(reinterpret_cast<const void*>(kq), shm_q, st) ||
      ma_host::reserve_lds(reinterpret_cast<const void*>(kk), shm_k, st))
    return 1;
  const int64_t streams = d->batch * d->num_heads * b.dil;
  a.tiles = (int32_t)((b.nr + QT - 1) / QT);
  ma_host::launch(false, kq, dim3((unsigned)(streams * a.tiles)), dim3(64 * NWQ), (uint32_t)shm_q, st, a);
  a.tiles = (int32_t)((b.nr + KT - 1) / KT);
  a.desc = 0;  // key tiles: the first see the most queries
  ma_host::launch(true, kk, dim3((unsigned)(streams * a.tiles)), dim3(64 * NWK), (uint32_t)shm_k, st, a);
  return 0;
}

// 4 waves and 64-row blocks (float32 above head_dim 64: 32-row): measured best
// of 4 or 8 waves and 32- or 64-row blocks (causal 128-key window, bf16,
// head_dim 128, 2 x 8 heads, 4096 rows: 74 us against 79-88; with P and dS in three
// planes 76).  Two workgroups a CU: registers for three cost more than they bring
// (same case, dQ 38 -> 41 us, dK/dV 35 -> 63).
//
// Causal rows in pairs of tiles, as in the forward: float32 above head_dim 32 on
// at most one 128-row tile per CU (8 heads of 4096 rows: head_dim 64 628 -> 561
// us, 128 1183 -> 981; 16-bit and narrow heads were 2-10 % slower), and 16-bit
// from saved statistics on half to one tile per CU (4096 rows: 138 -> 128 us).
//
// 16-bit at head_dim 64 from saved statistics (dense; P and dS rounded to 16
// bits, as in bwd_q_kernel / bwd_kv_kernel): blocks inside the band as
// straight-line code; with 256-row tiles enough for every CU (twice, for causal
// rows, whose tiles are uneven) two row groups per wave, so that each LDS read
// feeds two MFMAs.  8 heads, bwd_q + bwd_kv -> here: causal 2048 rows 77 -> 68 us,
// 8192 rows 339 -> 324, 16384 rows 1196 -> 980; all pairs, 8192 rows 629 -> 477.
// The longer tiles pay on long rows only (one group / two, bf16): causal 32 heads
// of 4096 rows 356 / 413 us, 16 of 8192 638 / 527; all pairs 400 heads of 600 rows
// 210 / 218, 64 of 1024 94 / 77; a 256-row tile of 64 rows is mostly idle (1024
// heads: 22 / 40).
template <typename T, int ND>
int bwd_nd(const ma_attn_desc* d, const FlArgs& a, hipStream_t st) {
  constexpr bool f32 = sizeof(T) == 4;
  constexpr int KB = f32 && ND > 2 ? 32 : 64;
  constexpr int NP = FlElt<T>::NPB;
  Band b;
  band_of(d, &b);
  const int64_t streams = d->batch * d->num_heads * b.dil;
  const int64_t tiles128 = streams * ((b.nr + 127) / 128), tiles256 = streams * ((b.nr + 255) / 256);
  FlArgs pair = a;
  pair.desc = 0;
  if constexpr (f32 && ND == 2) {  // saved statistics: head_dim 64
    if (a.fo) {
      if (a.desc && b.nr > 128 && tiles128 <= 256)
        return run_bwd<T, ND, 1, 1, 8, 8, KB, NP, 2, true, false, true>(d, pair, st);
      return run_bwd<T, ND, 1, 1, 4, 4, KB, NP, 2, true, false, false>(d, a, st);
    }
  }
  if constexpr (!f32 && ND == 2) {
    if (a.fo) {
      if (a.desc && tiles128 > 128 && tiles128 <= 256)
        return run_bwd<T, ND, 1, 1, 8, 8, KB, 1, 2, true, true, true>(d, pair, st);
      if (b.nr >= (a.desc ? 8192 : 1024) && tiles256 >= (a.desc ? 512 : 256))
        return run_bwd<T, ND, 2, 2, 8, 8, KB, 1, 2, true, true, false>(d, a, st);
      return run_bwd<T, ND, 1, 1, 4, 4, KB, 1, 3, true, true, false>(d, a, st);
    }
  }
  if constexpr (f32 && ND >= 2)
    if (a.desc && b.nr > 128 && tiles128 <= 256)
      return run_bwd<T, ND, 1, 1, 8, 8, KB, NP, 2, false, false, true>(d, pair, st);
  return run_bwd<T, ND, 1, 1, 4, 4, KB, NP, 2, false, false, false>(d, a, st);
}

template <typename T>
int bwd_t(const ma_attn_desc* d, const FlArgs& a, hipStream_t st) {
  switch ((d->head_dim + 31) / 32) {
    case 1: return bwd_nd<T, 1>(d, a, st);
    case 2: return bwd_nd<T, 2>(d, a, st);
    case 3: return bwd_nd<T, 3>(d, a, st);
    default: return bwd_nd<T, 4>(d, a, st);
  }
}

}  // namespace

bool applies(const ma_attn_desc* d, const void* const* ptrs, int n) {
  Band b;
  if (!band_of(d, &b) || d->head_dim < 8 || d->head_dim > 128 || d->head_dim % 8 != 0) return false;
  for (int i = 0; i < n; ++i)
    if (!aligned16(ptrs[i])) return false;
  const int64_t tb = b.dil * d->num_heads * d->head_dim * elt_of(d);
  // every byte offset a workgroup forms, the 16-row tiles' ids, and a launch's
  // 2^32 threads (64-row tiles of 256 and 128-row tiles of 512: many short
  // sequences reach it first)
  const int64_t streams = d->batch * d->num_heads * b.dil;
  return (b.nr + 512) * tb < (1LL << 31) && b.nr < (1LL << 29) && streams < (1LL << 31) &&
         streams * ((b.nr + 15) / 16) <= (int64_t)INT32_MAX && streams * ((b.nr + 63) / 64) < (1LL << 24) &&
         streams * ((b.nr + 127) / 128) < (1LL << 23);
}

int forward(const ma_attn_desc* d, const void* q, const void* k, const void* v, void* o, float* lse,
            hipStream_t st) {
  FlArgs a = args_of(d);
  a.q = q;
  a.k = k;
  a.v = v;
  a.o = o;
  a.lse = lse;
  switch (d->dtype) {
    case MA_ATTN_F32: return fwd_t<float>(d, a, st);
    case MA_ATTN_BF16: return fwd_t<__bf16>(d, a, st);
    default: return fwd_t<_Float16>(d, a, st);
  }
}

int forward_globals(const ma_attn_desc* d, int64_t num_global, const void* q, const void* k, const void* v, void* o,
                    hipStream_t st) {
  FlArgs a = args_of(d);
  a.q = q;
  a.k = k;
  a.v = v;
  a.o = o;
  a.globals = (int32_t)num_global;
  a.desc = 0;
  if (d->batch * d->num_heads * ((d->seq_len + 127) / 128) >= 256)
    return run_fwd<float, 2, 1, 8, 64, 2, FlElt<float>::NPB, true>(d, a, st);
  return run_fwd<float, 2, 1, 4, 64, 2, FlElt<float>::NPB, true>(d, a, st);
}

int backward(const ma_attn_desc* d, const void* const* ptrs, float* stats, const void* fo, const float* lse,
             hipStream_t st) {
  FlArgs a = args_of(d);
  a.q = ptrs[0];
  a.k = ptrs[1];
  a.v = ptrs[2];
  a.dout = ptrs[3];
  a.o = const_cast<void*>(ptrs[4]);
  a.dk = const_cast<void*>(ptrs[5]);
  a.dv = const_cast<void*>(ptrs[6]);
  a.stats = stats;
  a.fo = fo;
  a.lse = const_cast<float*>(lse);
  switch (d->dtype) {
    case MA_ATTN_F32: return bwd_t<float>(d, a, st);
    case MA_ATTN_BF16: return bwd_t<__bf16>(d, a, st);
    default: return bwd_t<_Float16>(d, a, st);
  }
}

}  // namespace ma_flash
