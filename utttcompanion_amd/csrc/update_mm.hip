// Backward pass and state write of one bf16 chunk update (reference fused_chunk_ttt_step,
// model/uttt_layer.py:279-534), gfx950 (MI355X): operands straight into LDS, fp32 state.
//
//   k_update_back   dH = dZ W_down^T per F tile, dU, dG, and the tile's squared gradient norm
//   k_update_write  one 64 x 64 gradient tile from the chunk's token slabs, then S' = beta S - c g,
//                   W' = decay W + S' (or only the tile's squared norm)
//
// The write is bound by the state it streams (48 D F bytes per row), the backward pass by the
// latency of its D loop on few workgroups.  Measured against the register-staged kernels they
// replaced (backward with the norm / state write with the row scalars, us):
//   1 row x 37 tokens, d 768, F 2048      28 -> 16 / 22 -> 14
//   8 rows x 64 tokens, d 768, F 2048     30 -> 20 / 146 -> 106 (604 MB, 5.7 TB/s)
//   4 rows x 64 tokens, d 2048, F 5504    91 -> 56 / 531 -> 398 (2.16 GB, 5.4 TB/s)
//   2 rows x 128 tokens, d 1024, F 2816   54 -> 25 / 147 -> 56
#include "update_mm.h"

#include "uttt_device.h"

namespace uttt {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // the caller's outputs: any fp32 alignment

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}
__device__ __forceinline__ void lds_write_b64(uint32_t addr, uint2 v) {
  asm volatile("ds_write_b64 %0, %1" ::"v"(addr), "v"(v));
}

// the four k pieces of rows rb .. rb + 31 of a row tile
__device__ __forceinline__ void row_frags(uint32_t tile, int rb, int lane, bf16x8 (&f)[4]) {
#pragma unroll
  for (int s = 0; s < 4; ++s) f[s] = lds_read_bf16x8<0>(row_frag_addr(tile, rb, lane, s));
}
template <int AHEAD>
__device__ __forceinline__ void wait_frags(bf16x8 (&f)[4]) {
  asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]) : "n"(AHEAD));
}
__device__ __forceinline__ void mma4(f32x16& acc, const bf16x8 (&a)[4], const bf16x8 (&b)[4]) {
#pragma unroll
  for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s], b[s], acc, 0, 0, 0);
}

// the eight transposing reads of a slab's fragments; slab_join after the wait makes the operands of them
__device__ __forceinline__ void slab_read(uint32_t addr, i16x4 (&r)[8]) {
  r[0] = lds_read_tr16<0>(addr);
  r[1] = lds_read_tr16<512>(addr);
  r[2] = lds_read_tr16<2048>(addr);
  r[3] = lds_read_tr16<2560>(addr);
  r[4] = lds_read_tr16<4096>(addr);
  r[5] = lds_read_tr16<4608>(addr);
  r[6] = lds_read_tr16<6144>(addr);
  r[7] = lds_read_tr16<6656>(addr);
}
template <int AHEAD>
__device__ __forceinline__ void slab_wait(i16x4 (&r)[8]) {
  asm volatile("s_waitcnt lgkmcnt(%8)"
               : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]), "+v"(r[6]), "+v"(r[7])
               : "n"(AHEAD));
}
__device__ __forceinline__ void slab_join(const i16x4 (&r)[8], bf16x8 (&f)[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k)
    f[k] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(r[2 * k], r[2 * k + 1], 0, 1, 2, 3, 4, 5, 6, 7));
}

__device__ __forceinline__ void lds_write_b16(uint32_t addr, bf16 v) {
  asm volatile("ds_write_b16 %0, %1" ::"v"(addr), "v"((uint32_t)__builtin_bit_cast(uint16_t, v)));
}

// One (F tile, row, token block).  NORM (one token block): then the tile's squared gradient norm, the
// sum of the squares of the gradient tiles K^T dU, K^T dG and dZ^T H, 64 x 64 each, in a second loop
// over D whose first slabs arrive while dU and dG are formed.  (Gram matrices, <K K^T, dU dU^T> and
// alike, need no second loop and took 14, 17 and 40 us at the first three shapes above, but their terms
// have both signs: 1e-6 relative on independent tokens, 1e-2 and more once a chunk's keys are nearly one.)
template <bool NORM>
__global__ void __launch_bounds__(kThreads, 2) k_update_back(const UpdateBackArgs a) {
  constexpr int SLOT = 2 * 8192;      // dZ rows by direct loads, W_down rows rounded through registers
  constexpr int PER = 2, WCH = 4;     // loads per wave and step, W_down pieces per thread
  constexpr int SLOTS = 3;
  __shared__ __align__(1024) char ring[SLOTS * SLOT];
  __shared__ __align__(1024) char slabs[NORM ? 3 * 8192 : 16];  // token slabs of H, dU, dG
  const int nF = a.F / 64;
  const RowTile rt = row_tile(blockIdx.x, a.B, nF * a.ntb);
  if (!rt.valid) return;
  const int b = rt.b, ft = rt.tile % nF, t0 = (rt.tile / nF) * 64, f0 = ft * 64;
  const int w = uniform((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32;
  const bf16* dz = static_cast<const bf16*>(a.dz) + ((int64_t)b * a.tok_pad + t0) * a.D;
  const float* wd = a.w_down + (int64_t)b * a.D * a.F + (int64_t)f0 * a.D;
  const int64_t rowbase = ((int64_t)b * a.tok_pad + t0) * a.F + f0;
  const uint32_t ring0 = lds_addr(ring), slab0 = lds_addr(slabs);

  int voff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) voff[i] = row_src_off(w + 4 * i, lane, a.D);
  auto issue = [&](int step, int at) {
    const uint32_t base = ring0 + (uint32_t)((at % SLOTS) * SLOT);
    const __amdgpu_buffer_rsrc_t rz = buffer_rsrc(dz + step * 64, (uint32_t)((64 * a.D - step * 64) * 2));
#pragma unroll
    for (int i = 0; i < 2; ++i)
      buffer_load_lds_raw(rz, lds_ptr(base + (uint32_t)((w + 4 * i) * 1024)), 16, voff[i], 0, 0, 0);
  };
  // W_down rows: thread's piece i is row 16 i + tid / 16, columns 4 (tid % 16) .. + 3
  struct Pieces {
    f32x4 r[WCH];
  };
  const int wrow = (int)threadIdx.x >> 4, wc4 = threadIdx.x & 15;
  const int wsrc = (wrow * a.D + 4 * wc4) * 4;
  const uint32_t wdst =
      ring0 + (uint32_t)(8192 + wrow * 128 + (((wc4 >> 1) ^ row_swz(wrow)) * 16) + (wc4 & 1) * 8);
  auto wload = [&](Pieces& p, int step) {
    const __amdgpu_buffer_rsrc_t r = buffer_rsrc(wd + step * 64, (uint32_t)(64 * a.D - step * 64) * 4u);
#pragma unroll
    for (int i = 0; i < WCH; ++i)
      p.r[i] =
          __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, wsrc, 16 * i * a.D * 4, 0));
  };
  auto wstore = [&](const Pieces& p, int step) {
    const uint32_t base = wdst + (uint32_t)((step % SLOTS) * SLOT);
#pragma unroll
    for (int i = 0; i < WCH; ++i)  // 16 rows on, the row's swizzle is the same
      lds_write_b64(base + (uint32_t)(i * 2048),
                    make_uint2(pack_bf16(p.r[i][0], p.r[i][1]), pack_bf16(p.r[i][2], p.r[i][3])));
  };

  if constexpr (NORM) {
    const __amdgpu_buffer_rsrc_t rh =
        buffer_rsrc(static_cast<const bf16*>(a.h) + rowbase, (uint32_t)((64 * a.F - f0) * 2));
#pragma unroll
    for (int i = 0; i < 2; ++i)
      buffer_load_lds_raw(rh, lds_ptr(slab0 + (uint32_t)((w + 4 * i) * 1024)), 16, slab_src_off(w + 4 * i, lane, a.F),
                          0, 0, 0);
  }
  const int nsteps = a.D / 64, last = nsteps - 1;
  Pieces p0, p1;
  wload(p0, 0);
  issue(0, 0);
  pin_loads();
  wload(p1, min(1, last));
  issue(min(1, last), 1);
  pin_loads();
  wstore(p0, 0);
  f32x16 dh;
  zero(dh);
  // loads run two steps ahead (the last steps load the last step again, so that every iteration has
  // the same loads in flight); a step's W_down pieces reach LDS during the step before it
  auto body = [&](int step, Pieces& mine, Pieces& next) {
    wait_vmcnt<WCH + PER>();
    asm volatile("s_waitcnt lgkmcnt(0)");
    __builtin_amdgcn_s_barrier();
    wload(mine, min(step + 2, last));
    issue(min(step + 2, last), step + 2);
    pin_loads();
    const uint32_t so = ring0 + (uint32_t)((step % SLOTS) * SLOT);
    bf16x8 fa[4], fb[4];
    row_frags(so, wr, lane, fa);
    row_frags(so + 8192u, wc, lane, fb);
    wait_frags<4>(fa);
    wait_frags<0>(fb);
    mma4(dh, fa, fb);
    __builtin_amdgcn_sched_barrier(0);
    wstore(next, step + 1);
  };
  int step = 0;
  for (; step + 2 <= nsteps; step += 2) {
    body(step, p0, p1);
    body(step + 1, p1, p0);
  }
  if (step < nsteps) body(step, p0, p1);
  float uv[16], gv[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int64_t off = rowbase + (int64_t)(wr + acc_row(i)) * a.F + wc + acc_col();
    uv[i] = a.u[off];
    gv[i] = a.g[off];
  }
  // the second loop's slabs: K, then dZ columns 64 step .. of the block's tokens
  auto issue_slabs = [&](int step) {
    const uint32_t base = ring0 + (uint32_t)((step % SLOTS) * SLOT);
    const bf16* kr = static_cast<const bf16*>(a.k) + (int64_t)b * a.k_rs + step * 64;
    // token rows past C read as zeros
    const __amdgpu_buffer_rsrc_t rk = buffer_rsrc(kr, (uint32_t)uniform((a.C * a.D - step * 64) * 2));
    const __amdgpu_buffer_rsrc_t rz = buffer_rsrc(dz + step * 64, (uint32_t)((64 * a.D - step * 64) * 2));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int off = slab_src_off(w + 4 * i, lane, a.D);
      buffer_load_lds_raw(rk, lds_ptr(base + (uint32_t)((w + 4 * i) * 1024)), 16, off, 0, 0, 0);
      buffer_load_lds_raw(rz, lds_ptr(base + 8192u + (uint32_t)((w + 4 * i) * 1024)), 16, off, 0, 0, 0);
    }
  };
  if constexpr (NORM) {
    wait_vmcnt<0>();  // the repeated loads
    asm volatile("s_waitcnt lgkmcnt(0)");
    __builtin_amdgcn_s_barrier();  // the ring is free
    for (int j = 0; j < min(nsteps, SLOTS - 1); ++j) issue_slabs(j);
  }
  const int f = wc + acc_col();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int t = wr + acc_row(i);
    const float u = uv[i], g = gv[i], sg = sigmoidf_acc(g);
    const bf16 du = from_f32<bf16>(dh[i] * (g * sg));
    const bf16 dg = from_f32<bf16>(dh[i] * u * (sg * (1.0f + g * (1.0f - sg))));
    const int64_t off = rowbase + (int64_t)t * a.F + f;
    static_cast<bf16*>(a.du)[off] = du;
    static_cast<bf16*>(a.dg)[off] = dg;
    if constexpr (NORM) {
      const uint32_t at = slab0 + (uint32_t)(t * 128 + (((f >> 3) ^ slab_swz(t)) * 16) + (f & 7) * 2);
      lds_write_b16(at + 8192u, du);
      lds_write_b16(at + 16384u, dg);
    }
  }
  if constexpr (NORM) {
    asm volatile("s_waitcnt lgkmcnt(0)");
    __builtin_amdgcn_s_barrier();  // dU, dG and H slabs are whole
    bf16x8 bu[4], bg[4], bh[4];
    {
      i16x4 ru[8], rg[8], rh[8];
      slab_read(slab_tr_addr(slab0 + 8192u, wc, lane), ru);
      slab_wait<0>(ru);
      slab_join(ru, bu);
      slab_read(slab_tr_addr(slab0 + 16384u, wc, lane), rg);
      slab_wait<0>(rg);
      slab_join(rg, bg);
      slab_read(slab_tr_addr(slab0, wc, lane), rh);
      slab_wait<0>(rh);
      slab_join(rh, bh);
    }
    const uint32_t tk = slab_tr_addr(ring0, wr, lane);
    float sq[4] = {0.f, 0.f, 0.f, 0.f};
    for (int step = 0; step < nsteps; ++step) {
      wait_steps<4, SLOTS - 2>(min(nsteps - 1, step + SLOTS - 2) - step);
      __builtin_amdgcn_s_barrier();  // the step's slabs are in LDS; the oldest slot is free
      if (step + SLOTS - 1 < nsteps) issue_slabs(step + SLOTS - 1);
      const uint32_t so = (uint32_t)((step % SLOTS) * SLOT);
      i16x4 rk[8], rz[8];
      slab_read(tk + so, rk);
      slab_read(tk + so + 8192u, rz);
      bf16x8 fk[4], fz[4];
      f32x16 gu, gg, gd;
      zero(gu);
      zero(gg);
      zero(gd);
      slab_wait<8>(rk);
      slab_join(rk, fk);
      mma4(gu, fk, bu);
      mma4(gg, fk, bg);
      slab_wait<0>(rz);
      slab_join(rz, fz);
      mma4(gd, fz, bh);
#pragma unroll
      for (int i = 0; i < 16; ++i) sq[i & 3] += gu[i] * gu[i] + gg[i] * gg[i] + gd[i] * gd[i];
    }
    const float total = block_sum((sq[0] + sq[1]) + (sq[2] + sq[3]), reinterpret_cast<float*>(ring));
    if (threadIdx.x == 0) a.nrm[b * nF + ft] = total;
  } else {
    wait_vmcnt<0>();  // the repeated loads
  }
}

// One 64 x 64 tile of one matrix: the gradient from the chunk's token slabs (tokens down the rows:
// transposing reads for both operands), then the state, whose 16-byte pieces were in flight
// meanwhile; the gradient tile crosses LDS so that they stay whole rows of 256 bytes.
//
// kNormOnly: only the tile's squared norm.  kScalarsGiven: the row scalars are read.  kFormScalars
// (one token block, F / 64 norm partials): every workgroup's first wave forms them while the slabs
// and the state are on their way.  Against a launch of their own in front, that is 1.9 us less for a
// 37-token chunk at d 768, F 2048 (of 55.7) and 25 us for eight chunks of 8 x 64 tokens (of 1519).
enum WriteForm { kNormOnly, kScalarsGiven, kFormScalars };

__device__ __forceinline__ float load_f32(const float* p, uint32_t bytes, int off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buffer_rsrc(p, bytes), off, 0, 0));
}

// The batch-global surprise, by one wave: masked token losses over all rows / valid tokens.
__device__ __forceinline__ void write_surprise(const UpdateWriteArgs& a, int lane) {
  float num = 0.f, den = 0.f;
  for (int b = 0; b < a.B; ++b) {
    num += a.loss[b * 64 + lane];
    if (lane < a.C) den += a.mask != nullptr ? a.mask[(int64_t)b * a.mask_rs + lane] : 1.f;
  }
  num = wave_sum(num);
  den = wave_sum(den);
  if (lane == 0) *a.surprise = a.mask != nullptr ? num / fmaxf(den, 1.f) : num / den;
}

template <WriteForm FORM>
__global__ void __launch_bounds__(kThreads) k_update_write(const UpdateWriteArgs a) {
  constexpr bool NORM = FORM == kNormOnly;
  constexpr int GLD = 68;  // floats per gradient tile row in LDS
  __shared__ __align__(1024) char ring[2 * 16384];  // two steps of one token block: A slab, B slab
  __shared__ float red[4];  // the norm's sum, or the row scalars
  static_assert(64 * GLD * 4 <= sizeof(ring), "the gradient tile reuses the ring");
  const int nD = a.D / 64, nF = a.F / 64, per = nD * nF;
  const RowTile rt = row_tile(blockIdx.x, a.B, 3 * per);
  if (!rt.valid) return;
  const int b = rt.b, m = rt.tile / per, j = rt.tile - m * per;
  const int w = uniform((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32;
  int r0, c0, ld_out, a_ld, b_ld, a_rows;
  const bf16 *as, *bs;
  if (m < 2) {  // W_up / W_gate tile (d, f) = K^T dU / K^T dG
    r0 = (j / nF) * 64;
    c0 = (j - (j / nF) * nF) * 64;
    ld_out = a.F;
    as = static_cast<const bf16*>(a.k) + (int64_t)b * a.k_rs + r0;
    a_ld = a.D;
    a_rows = a.C;
    bs = static_cast<const bf16*>(m == 0 ? a.du : a.dg) + (int64_t)b * a.tok_pad * a.F + c0;
    b_ld = a.F;
  } else {  // W_down tile (f, d) = H^T dZ
    r0 = (j / nD) * 64;
    c0 = (j - (j / nD) * nD) * 64;
    ld_out = a.D;
    as = static_cast<const bf16*>(a.h) + (int64_t)b * a.tok_pad * a.F + r0;
    a_ld = a.F;
    a_rows = a.tok_pad;  // rows past the chunk are zero
    bs = static_cast<const bf16*>(a.dz) + (int64_t)b * a.tok_pad * a.D + c0;
    b_ld = a.D;
  }
  const uint32_t ring0 = lds_addr(ring);
  int aoff[2], boff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    aoff[i] = slab_src_off(w + 4 * i, lane, a_ld);
    boff[i] = slab_src_off(w + 4 * i, lane, b_ld);
  }
  auto issue = [&](int tb) {
    const uint32_t base = ring0 + (uint32_t)((tb & 1) * 16384);
    const int rows = max(0, min(64, a_rows - 64 * tb));
    // the slabs' columns end 2 r0 (2 c0) bytes before their rows' next columns: ranges to the last row's end
    const __amdgpu_buffer_rsrc_t ra =
        buffer_rsrc(as + (int64_t)tb * 64 * a_ld, (uint32_t)uniform(rows > 0 ? (rows * a_ld - r0) * 2 : 0));
    const __amdgpu_buffer_rsrc_t rb = buffer_rsrc(bs + (int64_t)tb * 64 * b_ld, (uint32_t)((64 * b_ld - c0) * 2));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      buffer_load_lds_raw(ra, lds_ptr(base + (uint32_t)((w + 4 * i) * 1024)), 16, aoff[i], 0, 0, 0);
      buffer_load_lds_raw(rb, lds_ptr(base + 8192u + (uint32_t)((w + 4 * i) * 1024)), 16, boff[i], 0, 0, 0);
    }
  };
  // the first wave's pieces of the row scalars, loaded first (older than the loads the waits below
  // count) and without branches on lanes, which would wait for them here: lanes past a range read zeros
  float nrm0 = 0.f, nrm1 = 0.f, mask_v = 0.f, loss_v = 0.f;
  uint32_t alpha_v = 0;
  if constexpr (FORM == kFormScalars) {
    if (w == 0) {
      const float* nb = a.tile_nrm + (int64_t)b * nF;
      const uint32_t n_bytes = a.max_norm > 0.f ? (uint32_t)nF * 4u : 0u;
      nrm0 = load_f32(nb, n_bytes, 4 * lane);
      nrm1 = load_f32(nb, n_bytes, 4 * lane + 256);
      mask_v = load_f32(a.mask + (int64_t)b * a.mask_rs, a.mask != nullptr ? (uint32_t)a.C * 4u : 0u, 4 * lane);
      loss_v = load_f32(a.loss + b * 64, (uint32_t)a.C * 4u, 4 * lane);
      alpha_v = __builtin_amdgcn_raw_buffer_load_b16(
          buffer_rsrc(static_cast<const bf16*>(a.alpha) + (int64_t)b * a.alpha_rs, (uint32_t)a.C * 2u), 2 * lane, 0, 0);
    }
  }
  float clip = 0.f, decay = 0.f, act = 0.f;
  if constexpr (FORM == kScalarsGiven) {
    clip = a.scalars[4 * b];
    decay = a.scalars[4 * b + 1];
    act = a.scalars[4 * b + 2];
  }
  issue(0);
  if (a.ntb > 1) issue(1);
  pin_loads();
  // the state tile is the bulk of the traffic: its loads go out before the products
  const int64_t mat = (int64_t)a.D * a.F;
  const int row = (int)threadIdx.x >> 4, c4 = threadIdx.x & 15;
  const int64_t at = (int64_t)b * mat + (int64_t)(r0 + row) * ld_out + c0 + 4 * c4;
  f32x4 wv[4], sv[4];
  if constexpr (!NORM) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      wv[i] = *reinterpret_cast<const f32x4*>(a.w[m] + at + (int64_t)16 * i * ld_out);
      sv[i] = *reinterpret_cast<const f32x4*>(a.s[m] + at + (int64_t)16 * i * ld_out);
    }
  }
  pin_loads();  // eight of them for the first wait below
  if constexpr (FORM == kFormScalars) {
    if (w == 0) {
      float sq = nrm0 + nrm1;
      if (a.max_norm > 0.f)
        for (int i = lane + 128; i < nF; i += 64) sq += a.tile_nrm[b * nF + i];
      const float mt = a.mask != nullptr ? mask_v : lane < a.C ? 1.f : 0.f;
      asm volatile("" : "+v"(alpha_v));  // its widening stays here: beside the load it would wait there
      const float al = __builtin_bit_cast(float, alpha_v << 16);
      // squared norm, alpha, valid tokens, any valid, loss
      float sums[5] = {sq, a.mask != nullptr ? al * mt : al, mt, mt != 0.f ? 1.f : 0.f, loss_v};
#pragma unroll
      for (int i = 0; i < 5; ++i) sums[i] = wave_sum(sums[i]);
      if (lane == 0) {
        const float n = a.mask != nullptr ? fmaxf(sums[2], 1.f) : (float)a.C;
        const bool gated_off = a.min_row_surprise > 0.f && sums[4] / fmaxf(n, 1.f) < a.min_row_surprise;
        red[0] = a.max_norm > 0.f ? fminf(a.max_norm * (1.0f / sqrtf(sums[0] + 1e-8f)), 1.0f) : 1.0f;
        red[1] = 1.0f - sums[1] / n;
        red[2] = ((a.mask == nullptr || sums[3] > 0.f) && !gated_off) ? 1.f : 0.f;
        if (rt.tile == 0 && a.row_loss != nullptr) {
          a.row_loss[2 * b] = sums[4];
          a.row_loss[2 * b + 1] = sums[2];
        }
      }
    } else if (rt.tile == 0 && b == 0 && w == 3) {
      write_surprise(a, lane);
    }
  }
  f32x16 acc;
  zero(acc);
  const uint32_t ta = slab_tr_addr(ring0, wr, lane), tb0 = slab_tr_addr(ring0 + 8192u, wc, lane);
  for (int tb = 0; tb < a.ntb; ++tb) {
    if (tb == 0) {
      // block 0's loads are the oldest; block 1's and the state's may still be in flight
      if (a.ntb > 1)
        wait_vmcnt<NORM ? 4 : 12>();
      else
        wait_vmcnt<NORM ? 0 : 8>();
    } else {
      wait_vmcnt<0>();
    }
    __builtin_amdgcn_s_barrier();
    const uint32_t so = (uint32_t)((tb & 1) * 16384);
    bf16x8 fa[4], fb[4];
    slab_frags(ta + so, fa);
    slab_frags(tb0 + so, fb);
    lds_wait_frags(fa, fb);
    mma4(acc, fa, fb);
    if (tb + 2 < a.ntb) {
      __builtin_amdgcn_s_barrier();  // every wave is done with this slot
      issue(tb + 2);
    }
  }
  if constexpr (NORM) {
    float sq = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) sq += acc[i] * acc[i];
    const float total = block_sum(sq, red);
    if (threadIdx.x == 0) a.nrm[(int64_t)b * 3 * per + rt.tile] = total;
    return;
  }
  __builtin_amdgcn_s_barrier();  // the slabs are consumed: the gradient tile takes their place
  float* gt = reinterpret_cast<float*>(ring);
#pragma unroll
  for (int i = 0; i < 16; ++i) gt[(wr + acc_row(i)) * GLD + wc + acc_col()] = acc[i];
  __syncthreads();
  if constexpr (FORM == kFormScalars) {
    clip = red[0];
    decay = red[1];
    act = red[2];
  }
  const bool active = act != 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4 g = *reinterpret_cast<const f32x4*>(gt + (row + 16 * i) * GLD + 4 * c4);
    f32x4 wn, sn;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
      const float step = g[e] * clip;
      const float s_new = a.beta * sv[i][e] - step;
      const float w_new = decay * wv[i][e] + s_new;
      wn[e] = active ? w_new : wv[i][e];
      sn[e] = active ? s_new : sv[i][e];
    }
    *reinterpret_cast<f32x4u*>(a.w_out[m] + at + (int64_t)16 * i * ld_out) = wn;
    *reinterpret_cast<f32x4u*>(a.s_out[m] + at + (int64_t)16 * i * ld_out) = sn;
  }
}

}  // namespace

void launch_update_back(const UpdateBackArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)row_tile_blocks(a.B, (a.F / 64) * a.ntb));
  if (a.ntb == 1)
    hipLaunchKernelGGL(k_update_back<true>, grid, dim3(kThreads), 0, st, a);
  else
    hipLaunchKernelGGL(k_update_back<false>, grid, dim3(kThreads), 0, st, a);
}

static dim3 write_grid(const UpdateWriteArgs& a) {
  return dim3((unsigned)row_tile_blocks(a.B, 3 * (a.D / 64) * (a.F / 64)));
}

void launch_update_norm(const UpdateWriteArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(k_update_write<kNormOnly>, write_grid(a), dim3(kThreads), 0, st, a);
}

void launch_update_write(const UpdateWriteArgs& a, hipStream_t st) {
  if (a.scalars != nullptr)
    hipLaunchKernelGGL(k_update_write<kScalarsGiven>, write_grid(a), dim3(kThreads), 0, st, a);
  else
    hipLaunchKernelGGL(k_update_write<kFormScalars>, write_grid(a), dim3(kThreads), 0, st, a);
}

}  // namespace uttt
