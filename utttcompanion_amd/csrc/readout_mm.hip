// Matrix products of the frozen fast-weight readout over long token blocks (reference
// swiglu_fast_forward, model/uttt_layer.py:211-247, at prompt lengths), gfx950 (MI355X).
//
// Two products per batch row: H = SiLU(X W_gate) * (X W_up), then Z = H W_down.  X and H are
// token-major rows (k contiguous) and reach the MFMA's A operand as they are; W_up, W_gate
// (d rows) and W_down (f rows) have k down the rows and reach the B operand through transposing
// LDS reads, so no operand is transposed in memory.
//
// A workgroup takes MT tokens x 64 NS columns.  Per k step of 64 the row tiles and W slabs
// (8 KB each) go straight from global memory into one of SLOTS LDS slots while the previous step
// is consumed.  The gated product gives a wave 32 W_up columns and the same 32 W_gate columns,
// so that SwiGLU needs no exchange; the down product gives it 64 W_down columns.  fp32 W passes
// through registers, loaded up to two steps ahead and rounded to bf16 into the same slabs.
//
// What bounds them: wide tiles the matrix units and the operand reads out of L2 together (64 KB
// per 2048 MFMA cycles and CU; a library GEMM of this size reaches 1220-1420 TFLOP/s here), small
// shapes the latency of the first k steps.  Every operand descriptor is held in scalar registers:
// with ranges the compiler could not prove uniform, each load became a loop over the distinct
// descriptors of a wave (28 against 24 us at 1 x 333 tokens, d 768, F 2048).  Measured for the
// whole readout against the 64 x 64-tile kernels it replaced: 4 x 2048 tokens, d 2048, F 5504, bf16
// copies 1536 -> 561 us (988 TFLOP/s), fp32 masters 2524 -> 683 us; 2 x 333 tokens, d 768, F 2048
// 39 -> 28 us and 34 -> 33 us (there the down product is theirs still, see readout_mm_down); 128 tokens,
// d 2048, F 5504 52 -> 33 us and 60 -> 44 us.
#include "readout_mm.h"

#include <algorithm>

#include "uttt_device.h"

namespace uttt {
namespace {

// nseg row sets (segments) per batch row, rows_pad rows each (a multiple of 64, so a 64-row tile
// lies in one segment).  joint: one matrix of nseg rows_pad rows with segment 0's weights;
// otherwise each segment is a matrix of its own.
struct MmArgs {
  int B, nseg, joint;
  int rows, rows_pad, K, N;  // rows of A that exist, rows of the output per batch row and segment
  const bf16* a[2];          // (B, rows, K)
  int64_t a_rs[2];
  int a_ld;
  const void* w[2][2];  // per segment (B | 1, K, N): the two factors of the gated product, or W_down
  int64_t w_rs[2];
  int splits;
  int mtiles, ntiles;
  int rows_inner;  // tiles of all batch rows next to each other, as they read the same weights
  bf16* h[2];  // gated product: (B, rows_pad, N)
  float* u;    // gated product: segment 0's two factors' products, fp32 (B, rows_pad, N), or null
  float* g;
  float* zp;  // down product: (nseg, splits, B, rows_pad, N)
};

// LDS reads of one k piece of 16: MB A fragments (32 rows each, 4 KB apart) and 2 B fragments
template <int MB, int KK>
__device__ __forceinline__ void mm_read(bf16x8 (&fa)[MB], i16x4 (&fb)[4], uint32_t ta, uint32_t tb0, uint32_t tb1) {
  fa[0] = lds_read_bf16x8<0>(ta);
  if constexpr (MB > 1) fa[1] = lds_read_bf16x8<4096>(ta);
  if constexpr (MB > 2) {
    fa[2] = lds_read_bf16x8<8192>(ta);
    fa[3] = lds_read_bf16x8<12288>(ta);
  }
  fb[0] = lds_read_tr16<KK * 2048>(tb0);
  fb[1] = lds_read_tr16<KK * 2048 + 512>(tb0);
  fb[2] = lds_read_tr16<KK * 2048>(tb1);
  fb[3] = lds_read_tr16<KK * 2048 + 512>(tb1);
}

// wait until at most AHEAD later LDS reads are outstanding, tied to the fragments
template <int MB, int AHEAD>
__device__ __forceinline__ void mm_wait(bf16x8 (&fa)[MB], i16x4 (&fb)[4]) {
  if constexpr (MB == 4)
    asm volatile("s_waitcnt lgkmcnt(%8)"
                 : "+v"(fa[0]), "+v"(fa[1]), "+v"(fa[2]), "+v"(fa[3]), "+v"(fb[0]), "+v"(fb[1]), "+v"(fb[2]), "+v"(fb[3])
                 : "n"(AHEAD));
  else if constexpr (MB == 1)
    asm volatile("s_waitcnt lgkmcnt(%5)"
                 : "+v"(fa[0]), "+v"(fb[0]), "+v"(fb[1]), "+v"(fb[2]), "+v"(fb[3])
                 : "n"(AHEAD));
  else
    asm volatile("s_waitcnt lgkmcnt(%6)"
                 : "+v"(fa[0]), "+v"(fa[1]), "+v"(fb[0]), "+v"(fb[1]), "+v"(fb[2]), "+v"(fb[3])
                 : "n"(AHEAD));
}

template <int MB>
__device__ __forceinline__ void mm_mfma(f32x16 (&acc)[MB][2], const bf16x8 (&fa)[MB], const i16x4 (&fb)[4]) {
  const bf16x8 b0 = __builtin_bit_cast(bf16x8, __builtin_shufflevector(fb[0], fb[1], 0, 1, 2, 3, 4, 5, 6, 7));
  const bf16x8 b1 = __builtin_bit_cast(bf16x8, __builtin_shufflevector(fb[2], fb[3], 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], b0, acc[i][0], 0, 0, 0);
    acc[i][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], b1, acc[i][1], 0, 0, 0);
  }
}

__device__ __forceinline__ void lds_write_b64(uint32_t addr, uint2 v) {
  asm volatile("ds_write_b64 %0, %1" ::"v"(addr), "v"(v));
}

// WM x WN waves; a wave owns 32 MB rows and two 32-column blocks.
template <bool GATED, typename WT, int WM, int WN, int MB, int SLOTS>
__global__ void __launch_bounds__(WM* WN * 64) k_readout_mm(const MmArgs a) {
  constexpr int NW = WM * WN, NT = NW * 64;
  constexpr int MT = WM * MB * 32, RT = MT / 64;  // token rows, row tiles
  constexpr int NS = WN;                          // 64-column W slabs
  constexpr int SLOT = (RT + NS) * 8192;
  constexpr bool kDirect = sizeof(WT) == 2;  // bf16 W goes straight to LDS; fp32 through registers
  constexpr int GROUPS = (kDirect ? RT + NS : RT) * 8;
  static_assert(GROUPS % NW == 0, "a step's row groups split evenly over the waves");
  constexpr int PER = GROUPS / NW;
  constexpr int WCH = NS * 64 * 16 / NT;  // fp32 W: 16-byte pieces per thread and step
  __shared__ __align__(1024) char ring[SLOTS * SLOT];

  const int tile = xcd_contiguous(blockIdx.x, gridDim.x);
  int rest = tile;
  const int mt = rest % a.mtiles;
  rest /= a.mtiles;
  int bs = 0;
  if (a.rows_inner) {  // one segment
    bs = rest % a.B;
    rest /= a.B;
  }
  const int nt = rest % a.ntiles;
  rest /= a.ntiles;
  const int split = rest % a.splits;
  if (!a.rows_inner) bs = rest / a.splits;
  const int seg0 = bs / a.B, b = bs - seg0 * a.B;  // joint: always segment 0
  const int m0 = mt * MT, m_end = a.joint ? a.nseg * a.rows_pad : a.rows_pad;
  // a row of the matrix -> its segment, and where that begins
  auto seg_of = [&](int row) { return a.joint ? min(row / a.rows_pad, a.nseg - 1) : seg0; };
  auto seg_row = [&](int seg) { return a.joint ? seg * a.rows_pad : 0; };
  const int n0 = nt * (GATED ? 32 * NS : 64 * NS);  // first column of each factor
  const int steps_all = a.K / 64;
  const int s_begin = split * steps_all / a.splits, nsteps = (split + 1) * steps_all / a.splits - s_begin;

  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = w / WN, wn = w % WN;
  // slab sl holds columns n0 + 64 sl of W (down), or of W_up (sl < NS / 2) and W_gate
  auto slab_col = [&](int sl) { return n0 + 64 * (GATED ? sl % (NS / 2) : sl); };
  auto slab_src = [&](int sl) {
    return static_cast<const WT*>(a.w[seg0][GATED && sl >= NS / 2 ? 1 : 0]) + (int64_t)b * a.w_rs[seg0] +
           (int64_t)s_begin * 64 * a.N;
  };

  // wave w loads row groups w, w + NW, .. of a step: row tiles first, then slabs.  The sources and
  // ranges are wave-uniform by construction; said so, they stay in scalar registers
  int voff[PER];
  const char* src[PER];
  uint32_t bytes[PER];
  int64_t inc[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int g = w + NW * i, t = g >> 3;
    const bool is_row = !kDirect || t < RT;
    voff[i] = is_row ? row_src_off(g & 7, lane, a.a_ld) : slab_src_off(g & 7, lane, a.N);
    const int sl = is_row ? 0 : t - RT, c = slab_col(sl);
    // rows past the batch row's end read as zeros; columns past N read the next row (in range) or
    // zeros and are not stored
    const int row = m0 + 64 * t, seg = seg_of(row), lr = row - seg_row(seg);
    const bf16* rows = a.a[seg] + (int64_t)b * a.a_rs[seg] + (int64_t)lr * a.a_ld + (int64_t)s_begin * 64;
    const char* p = is_row ? reinterpret_cast<const char*>(rows) : reinterpret_cast<const char*>(slab_src(sl) + c);
    const uint32_t n = is_row ? (uint32_t)max(0, min(64, a.rows - lr)) * (uint32_t)a.a_ld * 2u
                              : (uint32_t)(64 * a.N - c) * 2u;
    const uint64_t u = reinterpret_cast<uint64_t>(p);
    src[i] = reinterpret_cast<const char*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)u) |
                                           (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(u >> 32)) << 32);
    bytes[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
    inc[i] = is_row ? 128 : (int64_t)64 * a.N * 2;
  }
  const uint32_t ring0 = lds_addr(ring);
  // step's tiles into the slot of `at`
  auto issue_at = [&](int step, int at) {
    const uint32_t base = ring0 + (uint32_t)((at % SLOTS) * SLOT);
#pragma unroll
    for (int i = 0; i < PER; ++i)
      buffer_load_lds_raw(buffer_rsrc(src[i] + step * inc[i], bytes[i]),
                          lds_ptr(base + (uint32_t)((w + NW * i) * 1024)), 16, voff[i], 0, 0, 0);
  };
  auto issue = [&](int step) { issue_at(step, step); };
  // fp32 W: this thread's pieces of a step in registers (4 columns each), then rounded into the slabs
  // thread: row NT / 16 k + tid / 16 of a slab, columns 4 (tid % 16) .. + 3
  constexpr int WROWS = NT / 16, WPS = 64 / WROWS;  // rows of a slab per pass, passes per slab
  struct WPieces {
    f32x4 r[kDirect ? 1 : WCH];
  };
  const int wrow = (int)threadIdx.x >> 4, wc4 = threadIdx.x & 15;
  const int wsrc = (wrow * a.N + 4 * wc4) * 4;
  const uint32_t wdst = ring0 + (uint32_t)(RT * 8192 + wrow * 128 + (((wc4 >> 1) ^ slab_swz(wrow)) * 16) + (wc4 & 1) * 8);
  auto wload = [&](WPieces& p, int step) {
#pragma unroll
    for (int i = 0; i < WCH; ++i) {
      const int sl = i / WPS, c = slab_col(sl);
      const __amdgpu_buffer_rsrc_t r =
          buffer_rsrc(slab_src(sl) + (int64_t)step * 64 * a.N + c, (uint32_t)(64 * a.N - c) * 4u);
      p.r[i] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, wsrc, (i % WPS) * WROWS * a.N * 4, 0));
    }
  };
  auto wstore = [&](const WPieces& p, int step) {
    const uint32_t base = wdst + (uint32_t)((step % SLOTS) * SLOT);
#pragma unroll
    for (int i = 0; i < WCH; ++i) {
      typedef float f32x2 __attribute__((ext_vector_type(2)));
      typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));
      uint2 v;
      v.x = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{p.r[i][0], p.r[i][1]}), bf16x2));
      v.y = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{p.r[i][2], p.r[i][3]}), bf16x2));
      // WROWS (16 or 32) rows on, the row's swizzle is the same
      lds_write_b64(base + (uint32_t)((i / WPS) * 8192 + (i % WPS) * WROWS * 128), v);
    }
  };

  // this wave's fragment addresses in slot 0
  const int rb = wm * MB * 32;
  uint32_t ta[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) ta[k] = row_frag_addr(ring0 + (uint32_t)((rb >> 6) * 8192), rb & 63, lane, k);
  const int sl0 = GATED ? wn / 2 : wn, sl1 = GATED ? NS / 2 + wn / 2 : wn;
  const int cb0 = GATED ? 32 * (wn & 1) : 0, cb1 = GATED ? 32 * (wn & 1) : 32;
  const uint32_t tb0 = slab_tr_addr(ring0 + (uint32_t)((RT + sl0) * 8192), cb0, lane);
  const uint32_t tb1 = slab_tr_addr(ring0 + (uint32_t)((RT + sl1) * 8192), cb1, lane);

  f32x16 acc[MB][2];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    zero(acc[i][0]);
    zero(acc[i][1]);
  }
  // the products of one step, its operands in LDS at slot offset so
  auto consume = [&](int step) {
    const uint32_t so = (uint32_t)((step % SLOTS) * SLOT);
    bf16x8 fa0[MB];
    i16x4 fb0[4];
    if constexpr (kDirect || MB < 4) {  // the next piece's reads are in flight during the products
      bf16x8 fa1[MB];
      i16x4 fb1[4];
      mm_read<MB, 0>(fa0, fb0, ta[0] + so, tb0 + so, tb1 + so);
      mm_read<MB, 1>(fa1, fb1, ta[1] + so, tb0 + so, tb1 + so);
      mm_wait<MB, MB + 4>(fa0, fb0);
      mm_mfma<MB>(acc, fa0, fb0);
      mm_read<MB, 2>(fa0, fb0, ta[2] + so, tb0 + so, tb1 + so);
      mm_wait<MB, MB + 4>(fa1, fb1);
      mm_mfma<MB>(acc, fa1, fb1);
      mm_read<MB, 3>(fa1, fb1, ta[3] + so, tb0 + so, tb1 + so);
      mm_wait<MB, MB + 4>(fa0, fb0);
      mm_mfma<MB>(acc, fa0, fb0);
      mm_wait<MB, 0>(fa1, fb1);
      mm_mfma<MB>(acc, fa1, fb1);
    } else {  // the registers hold the W pieces in flight instead
      mm_read<MB, 0>(fa0, fb0, ta[0] + so, tb0 + so, tb1 + so);
      mm_wait<MB, 0>(fa0, fb0);
      mm_mfma<MB>(acc, fa0, fb0);
      mm_read<MB, 1>(fa0, fb0, ta[1] + so, tb0 + so, tb1 + so);
      mm_wait<MB, 0>(fa0, fb0);
      mm_mfma<MB>(acc, fa0, fb0);
      mm_read<MB, 2>(fa0, fb0, ta[2] + so, tb0 + so, tb1 + so);
      mm_wait<MB, 0>(fa0, fb0);
      mm_mfma<MB>(acc, fa0, fb0);
      mm_read<MB, 3>(fa0, fb0, ta[3] + so, tb0 + so, tb1 + so);
      mm_wait<MB, 0>(fa0, fb0);
      mm_mfma<MB>(acc, fa0, fb0);
    }
  };
  if constexpr (kDirect) {
    for (int j = 0; j < min(nsteps, SLOTS - 1); ++j) issue(j);
    for (int step = 0; step < nsteps; ++step) {
      wait_steps<PER, SLOTS - 2>(min(nsteps - 1, step + SLOTS - 2) - step);
      __builtin_amdgcn_s_barrier();  // the step's operands are in LDS; the oldest slot is free
      if (step + SLOTS - 1 < nsteps) issue(step + SLOTS - 1);
      consume(step);
    }
  } else {
    // W pieces and rows are loaded AHEAD = SLOTS - 1 steps before use (the last steps load the
    // last step again, so that every iteration has the same loads in flight); a step's pieces are
    // written to its slot during the step before it
    constexpr int AHEAD = SLOTS - 1;
    static_assert(AHEAD == 1 || AHEAD == 2, "one or two register sets");
    const int last = nsteps - 1;
    WPieces p0, p1;
    wload(p0, 0);
    issue(0);
    pin_loads();
    if constexpr (AHEAD == 2) {
      wload(p1, min(1, last));
      issue_at(min(1, last), 1);
      pin_loads();
    }
    wstore(p0, 0);
    // the loads of step + AHEAD into `mine` (the pieces of `step`, stored already), then the
    // products, then the next step's pieces to LDS
    auto body = [&](int step, WPieces& mine, WPieces& next) {
      wait_vmcnt<(AHEAD - 1) * (WCH + PER)>();
      asm volatile("s_waitcnt lgkmcnt(0)");
      __builtin_amdgcn_s_barrier();
      wload(mine, min(step + AHEAD, last));
      issue_at(min(step + AHEAD, last), step + AHEAD);
      pin_loads();
      consume(step);
      __builtin_amdgcn_sched_barrier(0);  // no wait for the next pieces before the products are issued
      wstore(next, step + 1);
    };
    if constexpr (AHEAD == 1) {
      for (int step = 0; step < nsteps; ++step) body(step, p0, p0);
    } else {
      int step = 0;
      for (; step + 2 <= nsteps; step += 2) {
        body(step, p0, p1);
        body(step + 1, p1, p0);
      }
      if (step < nsteps) body(step, p0, p1);
    }
    wait_vmcnt<0>();  // the repeated loads
  }

  // acc[i][j][e]: row m0 + rb + 32 i + acc_row(e)
  const int n1 = n0 + (GATED ? 32 : 64) * wn;  // this wave's first column
  if (n1 >= a.N) return;
  const int col = n1 + acc_col();
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int row0 = m0 + rb + 32 * i;  // 32 rows of one segment
    if (row0 >= m_end) continue;
    const int seg = seg_of(row0), lr = row0 - seg_row(seg);
    if constexpr (GATED) {
      const int64_t base = ((int64_t)b * a.rows_pad + lr) * a.N + col;
      bf16* h = a.h[seg] + base;
      const bool keep = seg == 0 && a.u != nullptr;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float u = acc[i][0][e], g = acc[i][1][e];
        const int64_t off = (int64_t)acc_row(e) * a.N;
        h[off] = from_f32<bf16>((g * sigmoidf_acc(g)) * u);
        if (keep) {
          a.u[base + off] = u;
          a.g[base + off] = g;
        }
      }
    } else {
      float* z = a.zp + ((((int64_t)seg * a.splits + split) * a.B + b) * a.rows_pad + lr) * a.N + col;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        z[(int64_t)acc_row(e) * a.N] = acc[i][0][e];
        z[(int64_t)acc_row(e) * a.N + 32] = acc[i][1][e];
      }
    }
  }
}

int64_t ceil_div(int64_t x, int64_t y) { return (x + y - 1) / y; }

// Tile shapes: rows x columns (both factors of the gated product counted)
//   kWide   256 x 256, eight waves, one workgroup per CU
//   kMid    128 x 128, four waves
//   kSmall   64 x 128, four waves, two or three workgroups per CU
enum MmTile { kSmall, kMid, kWide };

int tile_rows(MmTile t) { return t == kWide ? 256 : t == kMid ? 128 : 64; }
int tile_cols(MmTile t) { return t == kWide ? 256 : 128; }

// Plan of one product: the tile shape (and for the down product the k split) of least time by
// this model, us: a round of the tiles that fit on the GPU together takes the k steps times the
// step's time of that shape, and a last partial round between a step's time at one workgroup per
// CU and that.  The step times are the fit to readouts timed with every tile shape and split
// forced, bf16 copies and fp32 masters, 100 to 16384 tokens at the model widths (d 512 to 2048);
// the plan is then within 6% of the best forced one on each of them.  Those of the gated product from
// fp32 W are the fit to that product alone over 290 readouts of 1 to 8 rows of 65 to 1500 tokens (0.2%
// from the best tile on average, 18% at most; with the down product's times 1.5% and 25%, and at 4 x 65
// tokens, d 1024, F 2816 the small tile's 26.0 us instead of the middle one's 23.8).  Wide tiles win where they
// fill the GPU, by reading each operand fewer times (4 x 2048 tokens, d 2048, F 5504, bf16: 950 /
// 778 / 700 us with H in small / mid / wide tiles, then 701 / 622 / 557 us with Z in them); smaller
// ones as soon as wide tiles leave CUs idle (2 x 333 tokens, d 768, F 2048: 32 / 35 / 48 us) or end
// in a nearly empty round (2048 tokens, d 2048, F 5504: 211 / 177 / 194 us, 344 wide tiles).
struct MmPlan {
  MmTile tile;
  int splits;
};

enum MmSteps { kBf16, kF32, kF32Readout };  // whose step times: kF32Readout the readout's gated product

MmPlan plan_mm(int64_t B, int64_t rows, int64_t cols, int64_t steps, int max_splits, MmSteps of) {
  constexpr double kFull[3][3] = {{0.87, 1.01, 1.89}, {1.40, 1.36, 2.30}, {1.40, 1.20, 2.10}};
  constexpr double kLone[3][3] = {{0.42, 0.90, 1.82}, {0.60, 1.02, 1.50}, {0.70, 0.90, 2.00}};
  constexpr int kPlaces[3] = {512, 512, 256}, kCus = 256;
  const double z_us = (double)B * rows * cols * 8.0 / 4e6;  // one more set of partials, written and read
  MmPlan best{kSmall, 1};
  double best_us = 1e300;
  for (int s = 1; s <= max_splits; ++s) {
    for (int t = kSmall; t <= kWide; ++t) {
      const MmTile tile = (MmTile)t;
      const int64_t n = B * ceil_div(rows, tile_rows(tile)) * ceil_div(cols, tile_cols(tile)) * s;
      const int64_t full = n / kPlaces[t], rest = n % kPlaces[t];
      const double k = (double)ceil_div(steps, s);
      double us = full * (k * kFull[of][t] + 2.0) + (s - 1) * z_us;
      if (rest > 0) {
        const double more = (double)std::max<int64_t>(0, rest - kCus) / kCus;
        us += k * (kLone[of][t] + more * (kFull[of][t] - kLone[of][t])) + 2.0;
      }
      if (us < best_us) {
        best_us = us;
        best = MmPlan{tile, s};
      }
    }
  }
  return best;
}

template <bool GATED, typename WT>
void launch_mm(MmArgs m, MmPlan p, hipStream_t st) {
  const int cols = GATED ? 2 * m.N : m.N;
  const int64_t matrices = m.joint ? m.B : (int64_t)m.B * m.nseg, rows = m.joint ? m.nseg * m.rows_pad : m.rows_pad;
  m.splits = p.splits;
  m.mtiles = (int)ceil_div(rows, tile_rows(p.tile));
  m.ntiles = (int)ceil_div(cols, tile_cols(p.tile));
  // Each XCD takes a contiguous eighth of the tile list and has its own L2.  Rows in turn make each XCD read
  // its rows' weights whole; where the rows share them and those are the larger operand, a weight tile's
  // tiles in turn make it read an eighth of them and all rows' tokens instead: 8 x 100 tokens through shared
  // fp32 W at d 768, F 2048 45.0 -> 38.8 us, 3 x 150 at d 1024, F 2816 50.0 -> 44.4 us.
  m.rows_inner = m.nseg == 1 && m.w_rs[0] == 0 && rows * m.B * 2 < (int64_t)cols * (int64_t)sizeof(WT);
  const dim3 grid((unsigned)(matrices * m.splits * m.mtiles * m.ntiles));
  if (p.tile == kWide)
    hipLaunchKernelGGL((k_readout_mm<GATED, WT, 2, 4, 4, 2>), grid, dim3(512), 0, st, m);
  else if (p.tile == kMid)
    hipLaunchKernelGGL((k_readout_mm<GATED, WT, 2, 2, 2, 2>), grid, dim3(256), 0, st, m);
  else
    hipLaunchKernelGGL((k_readout_mm<GATED, WT, 2, 2, 1, 3>), grid, dim3(256), 0, st, m);
}

constexpr int kMaxSplits = 8;
MmPlan plan_down(int64_t B, int64_t T, int64_t D, int64_t F, bool w_fp32) {
  return plan_mm(B, ceil_div(T, 64) * 64, D, F / 64, (int)std::min<int64_t>(kMaxSplits, F / 64),
                 w_fp32 ? kF32 : kBf16);
}

}  // namespace

int readout_mm_splits(int64_t B, int64_t T, int64_t D, int64_t F, bool w_fp32) {
  return plan_down(B, T, D, F, w_fp32).splits;
}

// From fp32 W the small tile is slower than k_down_partial's 64 x 64 one from 128 of those on, when two of
// them on a CU hide each other's loads: 3% with the LayerNorm over 122 readouts of 1 to 8 rows of 65 to
// 1500 tokens at the model widths, up to 18% (2 x 700 tokens at d 512: 12.2 against 9.1 us).  Below that it
// leaves fewer splits for the LayerNorm to sum: 4% faster over 94 of them.
bool readout_mm_down(int64_t B, int64_t T, int64_t D, int64_t F, bool w_fp32) {
  return !w_fp32 || B * ceil_div(T, 64) * (D / 64) < 128 || plan_down(B, T, D, F, true).tile != kSmall;
}

static MmPlan plan_update_down(int64_t B, int64_t T, int64_t D, int64_t F, bool joint, int most) {
  const int64_t rows = ceil_div(T, 64) * 64;
  return plan_mm(joint ? B : 2 * B, joint ? 2 * rows : rows, D, F / 64,
                 (int)std::min<int64_t>(std::min(most, kMaxSplits), F / 64), kF32);
}

int update_mm_splits(int64_t B, int64_t T, int64_t D, int64_t F, bool joint, int most) {
  return plan_update_down(B, T, D, F, joint, most).splits;
}

void launch_update_up(const UpdateMmArgs& a, bool joint, hipStream_t st) {
  MmArgs m{};
  m.B = a.B; m.nseg = 2; m.joint = joint; m.rows = a.T; m.rows_pad = a.tok_pad; m.K = a.D; m.N = a.F;
  m.a_ld = a.D;
  for (int s = 0; s < 2; ++s) {
    m.a[s] = static_cast<const bf16*>(a.x[s]); m.a_rs[s] = a.x_rs[s];
    m.w[s][0] = a.w_up[s]; m.w[s][1] = a.w_gate[s]; m.w_rs[s] = a.w_rs[s];
    m.h[s] = static_cast<bf16*>(a.h[s]);
  }
  m.u = a.u_store; m.g = a.g_store;
  launch_mm<true, float>(m, plan_mm(joint ? a.B : 2 * a.B, joint ? 2 * a.tok_pad : a.tok_pad, 2 * (int64_t)a.F,
                                    a.D / 64, 1, kF32), st);
}

void launch_update_down(const UpdateMmArgs& a, bool joint, hipStream_t st) {
  MmArgs z{};
  z.B = a.B; z.nseg = 2; z.joint = joint; z.rows = a.tok_pad; z.rows_pad = a.tok_pad; z.K = a.F; z.N = a.D;
  z.a_ld = a.F;
  for (int s = 0; s < 2; ++s) {
    z.a[s] = static_cast<const bf16*>(a.h[s]); z.a_rs[s] = (int64_t)a.tok_pad * a.F;
    z.w[s][0] = a.w_down[s]; z.w_rs[s] = a.w_rs[s];
  }
  z.zp = a.zp;
  launch_mm<false, float>(z, plan_update_down(a.B, a.T, a.D, a.F, joint, a.splits), st);
}

void launch_readout_up(const ReadoutMmArgs& a, hipStream_t st) {
  MmArgs m{};
  m.B = a.B; m.nseg = 1; m.rows = a.T; m.rows_pad = a.tok_pad; m.K = a.D; m.N = a.F;
  m.a[0] = static_cast<const bf16*>(a.x); m.a_rs[0] = a.x_rs; m.a_ld = a.D;
  m.w[0][0] = a.w_up; m.w[0][1] = a.w_gate; m.w_rs[0] = a.w_rs;
  m.h[0] = static_cast<bf16*>(a.h);
  const MmPlan p = plan_mm(a.B, a.tok_pad, 2 * (int64_t)a.F, a.D / 64, 1, a.w_fp32 ? kF32Readout : kBf16);
  if (a.w_fp32)
    launch_mm<true, float>(m, p, st);
  else
    launch_mm<true, bf16>(m, p, st);
}

void launch_readout_down(const ReadoutMmArgs& a, hipStream_t st) {
  MmArgs z{};
  z.B = a.B; z.nseg = 1; z.rows = a.tok_pad; z.rows_pad = a.tok_pad; z.K = a.F; z.N = a.D;
  z.a[0] = static_cast<const bf16*>(a.h); z.a_rs[0] = (int64_t)a.tok_pad * a.F; z.a_ld = a.F;
  z.w[0][0] = a.w_down; z.w_rs[0] = a.w_rs;
  z.zp = a.zp;
  const MmPlan p = plan_down(a.B, a.T, a.D, a.F, a.w_fp32);
  if (a.w_fp32)
    launch_mm<false, float>(z, p, st);
  else
    launch_mm<false, bf16>(z, p, st);
}

}  // namespace uttt
