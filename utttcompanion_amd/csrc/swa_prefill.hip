// Sliding-window GQA attention of prefill for bf16 operands, gfx950 (MI355X): flash-style, both
// products on v_mfma_f32_32x32x16_bf16.  Replaces the masked SDPA of the reference's prefill
// (model/uttt_layer.py:1119-1165); visibility rule :1028-1037.
//
// The work of one (row, kv head) is a list of units, one unit = 32 queries of one of its query
// heads, the heads of a 32-query block next to each other; a workgroup takes NW consecutive units,
// one per wave, which share each 64-key tile of K and V in LDS.  So the query heads of a kv head
// read its keys once together, and a tile's queries span only as many 32-query blocks as the
// waves need (a window of W keys costs a block W + 31 keys, where 64-query tiles cost W + 63).
//
// The scores are formed transposed, S^T = K Q^T (keys down the accumulator, one query per lane):
// the softmax of a query is then a reduction inside a lane and one exchange with the lane 32 away,
// rescaling is one multiplication per element by a per-lane factor, and the accumulator's layout
// is, after rounding, the B operand of O^T = V^T P^T as it is: lane half h holds keys 8 i + 4 h ..
// + 3 of each 16, and the V fragments are read in that key order.  K rows feed the A operand
// directly, V reaches it through transposing LDS reads; Q stays in registers.
//
// The running maximum is raised whenever a tile's scores exceed it, so that a query's heaviest weight
// is 1 exactly: the sum is formed from the unrounded weights, and a heaviest weight rounded to bf16
// would be off from its share of it.  (Raising it only past a factor of 2^8 saves most of the output's
// rescaling, 167 instead of 174 us for the first call below, and takes the relative error at scores of
// standard deviation 4 from 1.7e-3 to 2.1e-3.)
//
// What bounds it: LDS reads (each wave reads the whole K and V tile for its 32 queries, 32 KB per
// 1024 MFMA cycles at head_dim 128) about equal to the MFMAs, with the softmax's vector work between
// them.  Measured against the 16 x 16-tile kernel it replaced (64 queries per workgroup, V
// transposed through registers): 4 x 4096 queries, 16 heads on 4, head_dim 128, window 1024:
// 485 -> 174 us (690 TFLOP/s of visible pairs); 3 x 777 over 1288 keys, head_dim 64, window 512:
// 31.0 -> 19.4 us; one 64-token chunk of 4 rows over 1087 keys, head_dim 128, with the combine:
// 25.7 -> 19.2 us.
#include "swa_prefill.h"

#include <math.h>

#include <algorithm>

#include "uttt_device.h"

namespace uttt {
namespace {

constexpr int kQB = 32;  // queries per unit

struct SwaMmArgs {
  int n_kv_heads, rep, heads;
  int q_len, nqb, wgs;  // 32-query blocks, workgroups per (row, kv head) and split
  int nsplit, tiles_per_split, q_pad, groups;
  int64_t q_offset, kv_len, window;
  float scale, q_sign;  // scale > 0; Q enters times q_sign
  const bf16 *q, *k, *v;
  int64_t q_sb, q_sh, q_st, k_sb, k_sh, k_st, v_sb, v_sh, v_st;
  bf16* out;
  int64_t o_sb, o_sh, o_st;
  float* part;
};

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ const char* uniform(const void* p) {
  const uint64_t u = reinterpret_cast<uint64_t>(p);
  return reinterpret_cast<const char*>((uint64_t)(uint32_t)uniform((int)u) |
                                       (uint64_t)(uint32_t)uniform((int)(u >> 32)) << 32);
}

__device__ __forceinline__ float other_half(float x) { return __shfl_xor(x, 32, 64); }

// K fragments of one k step (dims 16 ks ..): keys 0-31 and 32-63 of the tile
template <int OFF>
__device__ __forceinline__ void k_read(bf16x8 (&f)[2], uint32_t addr) {
  f[0] = lds_read_bf16x8<OFF>(addr);
  f[1] = lds_read_bf16x8<OFF + 4096>(addr);
}
template <int AHEAD>
__device__ __forceinline__ void k_wait(bf16x8 (&f)[2]) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(f[0]), "+v"(f[1]) : "n"(AHEAD));
}

// V fragments of 16 keys (k step KS) for 32 NB output dims: addr[i] of dims 32 i ..
template <int NB, int KS>
__device__ __forceinline__ void v_read(i16x4 (&f)[2 * NB], const uint32_t (&addr)[NB], uint32_t so) {
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    f[2 * i] = lds_read_tr16<KS * 2048>(addr[i] + so);
    f[2 * i + 1] = lds_read_tr16<KS * 2048 + 1024>(addr[i] + so);
  }
}
template <int NB, int AHEAD>
__device__ __forceinline__ void v_wait(i16x4 (&f)[2 * NB]) {
  if constexpr (NB == 4)
    asm volatile("s_waitcnt lgkmcnt(%8)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7])
                 : "n"(AHEAD));
  else
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]) : "n"(AHEAD));
}
template <int NB>
__device__ __forceinline__ void pv_mfma(f32x16 (&o)[NB], const i16x4 (&f)[2 * NB], const bf16x8& p) {
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const bf16x8 vf =
        __builtin_bit_cast(bf16x8, __builtin_shufflevector(f[2 * i], f[2 * i + 1], 0, 1, 2, 3, 4, 5, 6, 7));
    o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, p, o[i], 0, 0, 0);
  }
}

template <int HD, int NW>
__global__ void __launch_bounds__(NW * 64, NW >= 6 ? 1 : 2) k_swa_prefill_mm(const SwaMmArgs a) {
  constexpr int NT = HD / 64;          // 64-dim tiles of K and of V per 64 keys
  constexpr int NB = HD / 32;          // 32-dim output blocks
  constexpr int KS = HD / 16;          // k steps of the scores
  constexpr int SLOT = 2 * NT * 8192;  // K tiles, then V slabs
  constexpr int GROUPS = 2 * NT * 8;   // 1 KB loads per key tile
  constexpr int PER = (GROUPS + NW - 1) / NW;  // per wave; past the last group a wave repeats one
  __shared__ __align__(1024) char ring[2 * SLOT];
  const RowTile rt = row_tile(blockIdx.x, a.groups, a.wgs * a.nsplit);
  if (!rt.valid) return;
  const int b = rt.b / a.n_kv_heads, kvh = rt.b - b * a.n_kv_heads;
  const int sp = rt.tile % a.nsplit, u0 = (rt.tile / a.nsplit) * NW;
  const int w = uniform((int)threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int units = a.rep * a.nqb;
  const int u = u0 + w, qb = min(u, units - 1) / a.rep;
  const int head = kvh * a.rep + u % a.rep;
  const bool unit_ok = u < units;

  // keys the workgroup's query blocks see, in tiles of 64 from the first one
  const int qb_first = u0 / a.rep, qb_last = min(u0 + NW - 1, units - 1) / a.rep;
  const int64_t lo = max((int64_t)0, a.q_offset + qb_first * kQB - a.window + 1);
  const int64_t hi = a.q_offset + min((int64_t)a.q_len, (int64_t)(qb_last + 1) * kQB);  // <= kv_len
  const int ntiles = (int)((hi - lo + 63) / 64);
  const int t_begin = sp * a.tiles_per_split, t_end = min(ntiles, t_begin + a.tiles_per_split);

  const int qi = qb * kQB + r;  // this lane's query
  const bool q_ok = unit_ok && qi < a.q_len;
  float* prow = a.part + ((((int64_t)b * a.heads + head) * a.nsplit + sp) * a.q_pad + qi) * (HD + 2);
  if (t_begin >= t_end) {  // nothing in this split's range (only with splits)
    if (q_ok && h == 0) {
      prow[0] = -INFINITY;
      prow[1] = 0.f;
    }
    return;
  }

  // Q fragments: query r, dims 16 s + 8 h .. + 7
  bf16x8 qf[KS];
  {
    const bf16* qr = a.q + b * a.q_sb + head * a.q_sh + (int64_t)qi * a.q_st + 8 * h;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (q_ok)
        qf[s] = *reinterpret_cast<const bf16x8*>(qr + 16 * s);
      else
        qf[s] = bf16x8{};
    }
    if (a.q_sign != 1.f) {
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[s][e] = from_f32<bf16>(to_f32((bf16)qf[s][e]) * a.q_sign);
    }
  }

  const bf16* kg = a.k + b * a.k_sb + kvh * a.k_sh;
  const bf16* vg = a.v + b * a.v_sb + kvh * a.v_sh;
  const uint32_t ring0 = lds_addr(ring);
  // wave w loads row groups w, w + NW, .. of a tile: K tiles first, then V slabs
  int voff[PER];
  const char* src[PER];
  int64_t row_bytes[PER];
  uint32_t dst[PER], early[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int g = (w + NW * i) % GROUPS, t = g >> 3;
    const bool is_k = t < NT;
    const int64_t st = is_k ? a.k_st : a.v_st;
    const int half = is_k ? t : t - NT;
    voff[i] = is_k ? row_src_off(g & 7, lane, (int)st) : slab_src_off(g & 7, lane, (int)st);
    src[i] = uniform((is_k ? kg : vg) + 64 * half);
    row_bytes[i] = (int64_t)uniform((int)(st * 2));
    early[i] = (uint32_t)uniform(128 * half);
    dst[i] = ring0 + (uint32_t)(g * 1024);
  }
  auto issue = [&](int t) {
    const int64_t kt0 = lo + (int64_t)t * 64;
    const int n = (int)min((int64_t)64, hi - kt0);  // keys past hi read as zeros
    const uint32_t so = (uint32_t)((t & 1) * SLOT);
#pragma unroll
    for (int i = 0; i < PER; ++i)
      buffer_load_lds_raw(buffer_rsrc(src[i] + kt0 * row_bytes[i], (uint32_t)uniform((int)(n * row_bytes[i] - early[i]))),
                          lds_ptr(dst[i] + so), 16, voff[i], 0, 0, 0);
  };

  uint32_t ka[4], va[NB];
#pragma unroll
  for (int s = 0; s < 4; ++s) ka[s] = row_frag_addr(ring0, 0, lane, s);
  {
    // transposing reads in the accumulator's key order: half h takes keys 4 h .. + 3, then 8 + 4 h ..
    const int g = lane >> 4, j16 = lane & 15, t = 4 * (g >> 1) + (j16 >> 2);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int c = 32 * (i & 1) + 16 * (g & 1) + 4 * (j16 & 3);
      va[i] = ring0 + (uint32_t)((NT + i / 2) * 8192 + t * 128 + (((c >> 3) ^ slab_swz(t)) * 16) + (c & 7) * 2);
    }
  }

  const float c2 = a.scale * 1.4426950408889634f;  // e^(scale s) = 2^(c2 s)
  float m = -INFINITY, l = 0.f;
  f32x16 o[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) zero(o[i]);

  const int64_t p_first = a.q_offset + (int64_t)qb * kQB;  // this wave's first and last query
  const int64_t p_last = a.q_offset + min((int64_t)a.q_len, (int64_t)(qb + 1) * kQB) - 1;
  const int win = (int)min(a.window, (int64_t)0x3fffffff);
  issue(t_begin);
  for (int t = t_begin; t < t_end; ++t) {
    wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();  // the tile is in LDS; every wave is done with the other slot
    if (t + 1 < t_end) issue(t + 1);
    const int64_t kt0 = lo + (int64_t)t * 64;
    if (!unit_ok || kt0 > p_last || kt0 + 63 <= p_first - a.window) continue;  // wave-uniform
    const uint32_t so = (uint32_t)((t & 1) * SLOT);

    f32x16 s[2];
    zero(s[0]);
    zero(s[1]);
    {
      bf16x8 f0[2], f1[2];
      auto mm = [&](const bf16x8(&f)[2], const bf16x8& q) {
        s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[0], q, s[0], 0, 0, 0);
        s[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[1], q, s[1], 0, 0, 0);
      };
      k_read<0>(f0, ka[0] + so);
      k_read<0>(f1, ka[1] + so);
      k_wait<2>(f0);
      mm(f0, qf[0]);
      k_read<0>(f0, ka[2] + so);
      k_wait<2>(f1);
      mm(f1, qf[1]);
      k_read<0>(f1, ka[3] + so);
      k_wait<2>(f0);
      mm(f0, qf[2]);
      if constexpr (HD == 64) {
        k_wait<0>(f1);
        mm(f1, qf[3]);
      } else {
        k_read<8192>(f0, ka[0] + so);
        k_wait<2>(f1);
        mm(f1, qf[3]);
        k_read<8192>(f1, ka[1] + so);
        k_wait<2>(f0);
        mm(f0, qf[4]);
        k_read<8192>(f0, ka[2] + so);
        k_wait<2>(f1);
        mm(f1, qf[5]);
        k_read<8192>(f1, ka[3] + so);
        k_wait<2>(f0);
        mm(f0, qf[6]);
        k_wait<0>(f1);
        mm(f1, qf[7]);
      }
    }
    if (kt0 + 63 > p_first || p_last - kt0 >= a.window) {  // an edge of the window crosses the tile
      const int rel = (int)(p_first - kt0) + r;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int d = rel - (32 * kb + acc_row(e));
          s[kb][e] = (unsigned)d < (unsigned)win ? s[kb][e] : -INFINITY;
        }
    }
    float tm = s[0][0];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) tm = fmaxf(tm, s[kb][e]);
    tm = fmaxf(tm, other_half(tm));
    if (__any(tm > m)) {
      const float m_new = fmaxf(m, tm);
      const float corr = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f((m - m_new) * c2);
      m = m_new;
      l *= corr;
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] *= corr;
    }
    const float base = m == -INFINITY ? 0.f : m * c2;
    bf16x8 p[4];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][e], c2, -base));
        l += x;
        p[2 * kb + (e >> 3)][e & 7] = from_f32<bf16>(x);
      }
    {
      i16x4 f0[2 * NB], f1[2 * NB];
      v_read<NB, 0>(f0, va, so);
      v_read<NB, 1>(f1, va, so);
      v_wait<NB, 2 * NB>(f0);
      pv_mfma<NB>(o, f0, p[0]);
      v_read<NB, 2>(f0, va, so);
      v_wait<NB, 2 * NB>(f1);
      pv_mfma<NB>(o, f1, p[1]);
      v_read<NB, 3>(f1, va, so);
      v_wait<NB, 2 * NB>(f0);
      pv_mfma<NB>(o, f0, p[2]);
      v_wait<NB, 0>(f1);
      pv_mfma<NB>(o, f1, p[3]);
    }
  }
  if (!q_ok) return;
  l += other_half(l);
  // o[i][e]: dim 32 i + 8 (e / 4) + 4 h + e % 4 of query r
  if (a.nsplit == 1) {
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    bf16* og = a.out + b * a.o_sb + head * a.o_sh + (int64_t)qi * a.o_st + 4 * h;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int e = 0; e < 16; e += 4) {
        bf16* d = og + 32 * i + 2 * e;
#pragma unroll
        for (int j = 0; j < 4; ++j) d[j] = from_f32<bf16>(o[i][e + j] * inv);
      }
  } else {
    if (h == 0) {
      prow[0] = m * a.scale;
      prow[1] = l;
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int e = 0; e < 16; e += 4) {
        float* d = prow + 2 + 32 * i + 2 * e + 4 * h;
#pragma unroll
        for (int j = 0; j < 4; ++j) d[j] = o[i][e + j];
      }
  }
}

constexpr int kMaxSplits = 16;

// Key splits so that about kWantedWgs workgroups of four units exist.  Splitting costs partials and a
// second launch (about 8 us), so it stops short of one workgroup per CU (timed before the running maximum
// was raised on every tile, which adds 4 to 8%): 3 x 777 queries over 1288
// keys (12 heads on 4, window 512), 228 workgroups of three waves: 17.9 us unsplit, 28.5 us in two;
// one 64-token chunk of 8 rows over 576 keys (64 workgroups): 13.7 us in three splits, 15.9 us in
// four; 4 rows of 64 tokens over 1088 keys, head_dim 128 (32 workgroups): 21 us in four to eight.
constexpr int kWantedWgs = 192;

int wanted_splits(int64_t batch, int64_t n_heads, int64_t q_len) {
  const int64_t units = batch * n_heads * ((q_len + kQB - 1) / kQB), wgs = (units + 3) / 4;
  return (int)std::max<int64_t>(1, std::min<int64_t>(kMaxSplits, (kWantedWgs + wgs - 1) / wgs));
}

// Eight units per workgroup (six where the heads come in threes, so that a workgroup's units fill
// whole query blocks) once that leaves a workgroup per CU: twice the waves share a tile's loads.
// Fewer units otherwise.
struct SwaPlan {
  int nw, wgs, nsplit, tiles_per_split;
};

SwaPlan plan_swa(const uttt_swa_prefill_args& a) {
  SwaPlan p;
  const int64_t rep = a.n_heads / a.n_kv_heads, nqb = (a.q_len + kQB - 1) / kQB, groups = a.batch * a.n_kv_heads;
  const int big = rep % 3 == 0 ? 6 : 8;
  const int64_t wgs_big = (rep * nqb + big - 1) / big;
  const bool use_big = groups * wgs_big >= 256;
  p.nw = use_big ? big : big / 2;
  p.wgs = (int)((rep * nqb + p.nw - 1) / p.nw);
  // query blocks a workgroup's units can touch, and the key tiles they can see
  const int64_t blocks = std::min<int64_t>(nqb, (p.nw - 1 + rep - 1) / rep + 1);
  const int64_t span = std::min<int64_t>(a.kv_len, std::min<int64_t>(a.window, a.kv_len) + blocks * kQB - 1);
  const int tiles = (int)((span + 63) / 64);
  const int ns = use_big ? 1 : std::min(tiles, wanted_splits(a.batch, a.n_heads, a.q_len));
  p.tiles_per_split = (tiles + ns - 1) / ns;
  p.nsplit = (tiles + p.tiles_per_split - 1) / p.tiles_per_split;
  return p;
}

template <int HD>
void launch(const SwaMmArgs& m, int nw, dim3 grid, hipStream_t st) {
  if (nw == 3)
    hipLaunchKernelGGL((k_swa_prefill_mm<HD, 3>), grid, dim3(192), 0, st, m);
  else if (nw == 4)
    hipLaunchKernelGGL((k_swa_prefill_mm<HD, 4>), grid, dim3(256), 0, st, m);
  else if (nw == 6)
    hipLaunchKernelGGL((k_swa_prefill_mm<HD, 6>), grid, dim3(384), 0, st, m);
  else
    hipLaunchKernelGGL((k_swa_prefill_mm<HD, 8>), grid, dim3(512), 0, st, m);
}

}  // namespace

int swa_prefill_mm_max_splits(int64_t batch, int64_t n_heads, int64_t q_len, int64_t kv_len, int64_t window) {
  const int64_t tiles = (std::min<int64_t>(kv_len, window) + 8 * kQB + 63) / 64;
  return (int)std::min<int64_t>(tiles, wanted_splits(batch, n_heads, q_len));
}

int swa_prefill_mm_splits(const uttt_swa_prefill_args& a) { return plan_swa(a).nsplit; }

void launch_swa_prefill_mm(const uttt_swa_prefill_args& a, float* part, int q_pad, hipStream_t st) {
  const SwaPlan p = plan_swa(a);
  SwaMmArgs m{};
  m.n_kv_heads = (int)a.n_kv_heads; m.heads = (int)a.n_heads; m.rep = (int)(a.n_heads / a.n_kv_heads);
  m.q_len = (int)a.q_len; m.nqb = (int)((a.q_len + kQB - 1) / kQB); m.wgs = p.wgs;
  m.nsplit = p.nsplit; m.tiles_per_split = p.tiles_per_split; m.q_pad = q_pad;
  m.groups = (int)(a.batch * a.n_kv_heads);
  m.q_offset = a.q_offset; m.kv_len = a.kv_len; m.window = a.window;
  // the kernel takes maxima of, and masks, the raw scores, which holds for a positive scale: Q carries
  // the sign of another one (exact in bf16), and for 0 the scores are 0 whatever their scale
  m.scale = a.scale != 0.f ? fabsf(a.scale) : 1.f;
  m.q_sign = a.scale > 0.f ? 1.f : a.scale < 0.f ? -1.f : 0.f;
  m.q = static_cast<const bf16*>(a.q); m.k = static_cast<const bf16*>(a.k); m.v = static_cast<const bf16*>(a.v);
  m.q_sb = a.q_stride_b; m.q_sh = a.q_stride_h; m.q_st = a.q_stride_t;
  m.k_sb = a.k_stride_b; m.k_sh = a.k_stride_h; m.k_st = a.k_stride_t;
  m.v_sb = a.v_stride_b; m.v_sh = a.v_stride_h; m.v_st = a.v_stride_t;
  m.out = static_cast<bf16*>(a.out);
  m.o_sb = a.o_stride_b; m.o_sh = a.o_stride_h; m.o_st = a.o_stride_t;
  m.part = part;
  const dim3 grid((unsigned)row_tile_blocks(m.groups, p.wgs * p.nsplit));
  if (a.head_dim == 64)
    launch<64>(m, p.nw, grid, st);
  else
    launch<128>(m, p.nw, grid, st);
}

}  // namespace uttt
