// codec.hip -- HIP kernels of the RVQ codec decode (crates/fish_s2_infer/src/codec.rs:1690-1714).
//
// The decoder's convolutions (causal conv1d, transposed conv1d, pointwise
// linears) all run on one implicit-GEMM MFMA kernel, conv_gemm_kernel:
//   * block tile: 128 frames x 192 or 256 output channels (4 waves in 2 x 2) or
//     256 frames x 96 (4 x 1), each wave 64 frames x 96 or 128 channels of
//     v_mfma_f32_32x32x16_f16 (frames as the A operand, weights as B, so the 32
//     lanes of a row group store 32 consecutive channels of one frame);
//   * K runs over stages of 32 input channels and, in a stage, over the taps:
//     a stage holds the window of the tile's frames plus the halo the taps
//     reach back, read by every tap at its own row offset; a step holds one
//     tap's weights for those channels;
//   * activations and weights lie in memory as contiguous KiB tiles of 16 rows
//     x 32 channels, staged by LDS-DMA loads of one KiB per wave: weights NB
//     steps ahead, windows NA stages ahead.  (Frame-major rows were read 32
//     bytes at a time into registers, one stage ahead.)  The causal padding is
//     a zeroed guard before each plane, so no load is predicated;
//   * a step is computed in two halves of 16 channels; the next half's
//     fragments are read from LDS while the current one multiplies, and the
//     barrier between the halves frees the step's buffers;
//   * tiles of one weight tile (m tile) are dealt to the same XCD, so that
//     XCD's L2 serves its weights to all of its frame tiles.
// Measured at 2048 latent frames (512 code frames; before: 256-frame tiles of
// 16-channel stages through registers), us: entry 78 -> 71, transposed convs of
// blocks 1-4 238 / 448 / 621 / 441 -> 141 / 313 / 387 / 304, k7 convs of blocks 1
// and 2 184 / 346 -> 128 / 258, their k1 convs 91 / 232 -> 43 / 152, a residual unit
// of block 3 (k7 and k1 in one launch now) 856 -> 472, of block 4 548 -> 359;
// whole decode 10.34 -> 7.02 ms.
// Small per-frame kernels handle the rest: RVQ lookup, the windowed attention of
// the post-module transformer (RoPE as it reads q and k), depthwise conv +
// LayerNorm, the output conv + tanh.

#include <algorithm>

#include "codec.h"
#include "expf_glibc.h"
#include "launch.h"
#include "lds_dma.h"
#include "wave.h"
#include "sin_cw.h"

namespace s2 {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr size_t CG_FMAJOR_WEIGHT_BYTES = size_t(3) << 19;  // 1.5 MiB of a 4 MiB XCD L2

// swizzle of a 16-row activation tile (act_off): the 16-byte chunk c of row r
// sits at c ^ act_swz(r), so 16 consecutive rows from any start put one chunk
// each on distinct LDS banks
__device__ __forceinline__ uint32_t act_swz(uint32_t r) { return ((r >> 1) & 3u) ^ ((r >> 3) & 1u); }
// offset in halfs of channel c of frame f in a plane of C channels
__device__ __forceinline__ size_t act_off(uint32_t f, uint32_t c, uint32_t C) {
  return (size_t(f >> 4) * (C >> 5) + (c >> 5)) * 512 + (f & 15u) * 32u + ((((c >> 3) & 3u) ^ act_swz(f)) << 3) +
         (c & 7u);
}

// erf_approx and gelu_erf (codec.rs:3886-3899), the reference's operation order.
__device__ __forceinline__ float erf_as(float value) {
  const float sign = value < 0.0f ? -1.0f : 1.0f;
  const float x = fabsf(value);
  const float t = __fdiv_rn(1.0f, __fadd_rn(1.0f, __fmul_rn(0.3275911f, x)));
  float p = __fsub_rn(__fmul_rn(1.0614054f, t), 1.4531521f);
  p = __fadd_rn(__fmul_rn(p, t), 1.4214138f);
  p = __fsub_rn(__fmul_rn(p, t), 0.28449672f);
  p = __fadd_rn(__fmul_rn(p, t), 0.2548296f);
  p = __fmul_rn(p, t);
  return __fmul_rn(sign, __fsub_rn(1.0f, __fmul_rn(p, expf_glibc(__fmul_rn(-x, x)))));
}
__device__ __forceinline__ float gelu_as(float v) {
  return __fmul_rn(__fmul_rn(0.5f, v), __fadd_rn(1.0f, erf_as(__fmul_rn(v, 0.70710677f))));
}
// snake_activation_frame_major (codec.rs:2162-2186), sin^2 from sin_cw.h;
// inv = 1 / (guarded alpha), once per channel
__device__ __forceinline__ float snake(float x, float alpha, float inv) { return snake_cw(x, alpha, inv); }

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); }

template <int G, int PL, int MC, int FC, int WMG, int NB, int NA, bool FU, int OS>
__global__ __launch_bounds__(256, 2) void conv_gemm_kernel(ConvGemmArgs a, uint32_t m_tiles, uint32_t f_tiles,
                                                           int32_t tile0, uint32_t a_tiles, int32_t t0, int32_t tstep,
                                                           uint32_t fmajor) {
  constexpr uint32_t MT = 32 * MC * WMG, FT = 32 * FC * (4 / WMG);
  constexpr uint32_t AT = FT / 16 + (G == 7 ? 4 : G == 1 ? 0 : 1);  // most 16-frame tiles of a window
  constexpr uint32_t WSTEP = MT * 64, APL = AT * 1024, ABUF = PL * APL;
  constexpr int PW = (int(MT / 16) + 3) / 4, PA = (PL * int(AT) + 3) / 4;  // KiB loads per wave
  extern __shared__ __align__(16) uint8_t cg_lds[];
  const uint32_t lane = threadIdx.x & 63u, wave = uniform(threadIdx.x >> 6);
  const uint32_t wm = wave % WMG, wf = wave / WMG;
  // Workgroup b runs on XCD b % 8; tiles are dealt to XCDs in contiguous
  // ranges (XCD-major), in one of two orders.
  //   fmajor: over all phases, t = (ft * phases + phase) * m_tiles + mt, so
  //     the blocks that read one frame tile's input window (every phase and
  //     weight tile) run one after another on one XCD: the window comes from
  //     HBM once and from that XCD's L2 after, while the weights of every
  //     (phase, m tile), small enough, stay in each L2.
  //   otherwise: phase by phase (phase = b / (m_tiles f_tiles)), and within
  //     a phase t = mt * f_tiles + ft: an XCD works through one weight tile at
  //     a time, which its L2 serves to all of that XCD's frame tiles.
  const uint32_t nb1 = m_tiles * f_tiles;
  uint32_t b = blockIdx.x, nb = gridDim.x, phase = 0, phases = nb / nb1;
  if (!fmajor) {
    phase = b / nb1;
    b -= phase * nb1;
    nb = nb1;
  }
  const uint32_t xcd = b & 7u, slot = b >> 3, q8 = nb >> 3, r8 = nb & 7u;
  const uint32_t t = xcd < r8 ? xcd * (q8 + 1u) + slot : r8 * (q8 + 1u) + (xcd - r8) * q8 + slot;
  uint32_t mt, ft;
  if (fmajor) {
    mt = t % m_tiles;
    const uint32_t tr = t / m_tiles;
    phase = tr % phases;
    ft = tr / phases;
  } else {
    mt = t / f_tiles;
    ft = t - mt * f_tiles;
  }
  // (the divisions above are expanded on the vector unit: move the results
  // to scalar registers, where they cost no vector registers in the loop)
  mt = uniform(mt);
  ft = uniform(ft);
  phase = uniform(phase);
  const uint32_t f0 = ft * FT, kt = a.C / 32, splits = gridDim.z, sp = blockIdx.z;
  const int32_t c0 = int32_t(kt * sp / splits), c1 = int32_t(kt * (sp + 1) / splits);
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(cg_lds)), off = lane * 16u;

  // this wave's loads: weight tiles PW wave + j of a step, activation tiles
  // PA wave + j of a window (plane-major); a load past the last tile repeats it
  const uint8_t* wsrc = reinterpret_cast<const uint8_t*>(a.w) + (size_t(phase) * m_tiles + mt) * (size_t(G) * WSTEP * kt);
  const uint8_t* asrc[PA];
  uint32_t adst[PA];
#pragma unroll
  for (int j = 0; j < PA; ++j) {
    const uint32_t q = min(PA * wave + j, uint32_t(PL) * AT - 1u), plane = q / AT, tile = min(q % AT, a_tiles - 1u);
    asrc[j] = reinterpret_cast<const uint8_t*>(plane ? a.xl : a.xh) +
              (int64_t(f0 / 16u) + tile0 + int32_t(tile)) * int64_t(kt) * 1024;
    adst[j] = lds0 + NB * WSTEP + plane * APL + tile * 1024u;
  }
  auto issue_w = [&](int32_t idx, uint32_t buf) {  // step idx = stage * G + tap, from this split's first
    const uint8_t* src = wsrc + size_t(min(idx, (c1 - c0) * G - 1) + c0 * G) * WSTEP;
#pragma unroll
    for (int j = 0; j < PW; ++j) {
      const uint32_t q = min(PW * wave + j, MT / 16u - 1u) * 1024u;
      dma16(src + q, off, lds0 + buf + q);
    }
  };
  auto issue_a = [&](int32_t st, uint32_t buf) {
    const uint32_t k = uint32_t(min(c0 + st, c1 - 1)) * 1024u;
#pragma unroll
    for (int j = 0; j < PA; ++j) dma16(asrc[j] + k, off, adst[j] + buf);
  };

  const uint32_t fr = lane & 31u;
  const uint32_t wrd = wm * MC * 2048u + (fr >> 4) * 1024u + (fr & 15u) * 16u + (lane >> 5) * 256u;
  const uint32_t arow = wf * 32u * FC + fr;
  struct Frags {
    half8 w[MC], x[FC][PL];
  };
  auto read = [&](Frags& f, uint32_t wbuf, uint32_t abuf, int g, uint32_t h) {
    const uint32_t row = arow + uint32_t(t0 + g * tstep);
    const uint8_t* pa = cg_lds + abuf + row * 64u + (((2u * h + (lane >> 5)) ^ act_swz(row)) << 4);
#pragma unroll
    for (int i = 0; i < FC; ++i)
#pragma unroll
      for (int p = 0; p < PL; ++p) f.x[i][p] = *reinterpret_cast<const half8*>(pa + p * APL + i * 2048);
    const uint8_t* pw = cg_lds + wbuf + wrd + h * 512u;
#pragma unroll
    for (int j = 0; j < MC; ++j) f.w[j] = *reinterpret_cast<const half8*>(pw + j * 2048);
  };
  // 32-frame waves have the registers for sums in two levels: every FL stages (16 to
  // 28 roundings) acc goes into sum and starts again from zero.  They serve the
  // launches of few blocks, where 256-frame tiles split the input channels up to 8
  // ways and so kept every running sum short; these tiles split less, and the
  // entry conv of 700 frames was 2.7e-7 off 64 bits instead of 2.0e-7 (with this
  // 1.5e-7, for 1 to 2 % of a decode of up to 260 code frames).
  constexpr bool TWO = FC == 1;
  constexpr int FL = G == 1 ? 4 : 2;
  floatx16 acc[FC][MC], sum[TWO ? FC : 1][TWO ? MC : 1];
#pragma unroll
  for (int i = 0; i < FC; ++i)
#pragma unroll
    for (int j = 0; j < MC; ++j) {
      acc[i][j] = floatx16{};
      if constexpr (TWO) sum[i][j] = floatx16{};
    }
  auto mma = [&](const Frags& f) {
#pragma unroll
    for (int p = 0; p < PL; ++p)
#pragma unroll
      for (int j = 0; j < MC; ++j)
#pragma unroll
        for (int i = 0; i < FC; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.x[i][p], f.w[j], acc[i][j], 0, 0, 0);
  };
  constexpr uint32_t A0 = NB * WSTEP;  // LDS byte of the first window
  // The loads go out in the order of the steps that issue them (below), from
  // as many steps before the first as the buffers reach ahead.
  constexpr int PRE = NB > NA * G ? NB : NA * G;
#pragma unroll
  for (int v = -PRE; v < 0; ++v) {
    if ((v + PRE * G) % G == G - 1 && (v - (G - 1)) / G + NA >= 0) {
      const int st = (v - (G - 1)) / G + NA;
      issue_a(st, (st % NA) * ABUF);
    }
    if (v + NB >= 0) issue_w(v + NB, ((v + NB) % NB) * WSTEP);
  }
  __builtin_amdgcn_s_waitcnt(wait_imm(0, false));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags fa, fb;
  uint32_t wbuf = 0, abuf = A0;
  int32_t idx = 0;
  read(fa, wbuf, abuf, 0, 0);
  for (int32_t st = 0; st < c1 - c0; ++st) {
#pragma unroll
    for (int g = 0; g < G; ++g, ++idx) {
      read(fb, wbuf, abuf, g, 1);
      __builtin_amdgcn_sched_barrier(0);
      mma(fa);
      __builtin_amdgcn_sched_barrier(0);
      // Wait for the weights of step idx + 1 (and, at the last tap, the next
      // window): NB - 2 later weight steps may be in flight and the windows
      // issued among them; lgkmcnt(0): this step's buffers are read.
      constexpr auto later = [](int gg) {
        int n = (NB - 2) * PW;
        for (int k = 0; k <= NB - 3; ++k) n += k % G == gg % G ? PA : 0;
        const int na = (NA - 1) * G * PW + (NA - 2) * PA;
        return gg == G - 1 && na < n ? na : n;
      };
      switch (g) {  // (a constant after unrolling; the immediate must be one)
        case 0: __builtin_amdgcn_s_waitcnt(wait_imm(later(0), true)); break;
        case 1: __builtin_amdgcn_s_waitcnt(wait_imm(later(1), true)); break;
        case 2: __builtin_amdgcn_s_waitcnt(wait_imm(later(2), true)); break;
        case 3: __builtin_amdgcn_s_waitcnt(wait_imm(later(3), true)); break;
        case 4: __builtin_amdgcn_s_waitcnt(wait_imm(later(4), true)); break;
        case 5: __builtin_amdgcn_s_waitcnt(wait_imm(later(5), true)); break;
        default: __builtin_amdgcn_s_waitcnt(wait_imm(later(6), true)); break;
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (g == G - 1) {
        issue_a(st + NA, abuf - A0);
        abuf = abuf + ABUF == A0 + NA * ABUF ? A0 : abuf + ABUF;
      }
      issue_w(idx + NB, wbuf);
      wbuf = wbuf + WSTEP == NB * WSTEP ? 0u : wbuf + WSTEP;
      read(fa, wbuf, abuf, g == G - 1 ? 0 : g + 1, 0);
      __builtin_amdgcn_sched_barrier(0);
      mma(fb);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (TWO) {
      if ((st + 1) % FL == 0) {
#pragma unroll
        for (int i = 0; i < FC; ++i)
#pragma unroll
          for (int j = 0; j < MC; ++j) {
            sum[i][j] += acc[i][j];
            acc[i][j] = floatx16{};
          }
      }
    }
  }
  if constexpr (TWO) {
#pragma unroll
    for (int i = 0; i < FC; ++i)
#pragma unroll
      for (int j = 0; j < MC; ++j) acc[i][j] = sum[i][j] + acc[i][j];
  }
  // the unused tail loads have landed before LDS is used again or the block ends
  __builtin_amdgcn_s_waitcnt(wait_imm(0, true));

  if constexpr (FU) {
    // The residual unit's k1 conv on the tile just computed (all M channels):
    // Y = f16(snake(acc + bias_mid, alpha_mid)) in LDS ([32 channels][frame][64
    // bytes], swizzled like a window); its weights go straight to registers
    // from the fragment-ordered copy, a step ahead.
    const uint8_t* w1 = reinterpret_cast<const uint8_t*>(a.w1) + wrd;
    half8 wn[2][MC];
    auto load_w1 = [&](uint32_t c) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < MC; ++j) wn[h][j] = *reinterpret_cast<const half8*>(w1 + c * WSTEP + h * 512u + j * 2048);
    };
    load_w1(0);
    __syncthreads();  // every wave's tail loads have landed
#pragma unroll
    for (int j = 0; j < MC; ++j) {
      const uint32_t m = (wm * MC + j) * 32u + fr;
      const float bm = a.bias_mid[m], am = snake_guard(a.alpha_mid[m]), im = 1.0f / am;
      uint8_t* yc = cg_lds + (m >> 5) * (FT * 64u) + (m & 7u) * 2u;
#pragma unroll
      for (int i = 0; i < FC; ++i) {
        const uint32_t fl = wf * 32u * FC + i * 32u + 4u * (lane >> 5);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const uint32_t row = fl + 8u * (v >> 2) + (v & 3);
          const float val = snake(__fadd_rn(acc[i][j][v], bm), am, im);
          *reinterpret_cast<_Float16*>(yc + row * 64u + ((((m >> 3) & 3u) ^ act_swz(row)) << 4)) = _Float16(val);
          acc[i][j][v] = 0.0f;
          if (v % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t c = 0; c < MT / 32; ++c) {
      half8 w[2][MC], x[2][FC];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < MC; ++j) w[h][j] = wn[h][j];
#pragma unroll
        for (int i = 0; i < FC; ++i)
          x[h][i] = *reinterpret_cast<const half8*>(cg_lds + c * (FT * 64u) + (arow + 32u * i) * 64u +
                                                    (((2u * h + (lane >> 5)) ^ act_swz(arow)) << 4));
      }
      if (c + 1 < MT / 32) load_w1(c + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < MC; ++j)
#pragma unroll
          for (int i = 0; i < FC; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[h][i], w[h][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  if (splits > 1) {  // partial sums; conv_split_reduce_kernel finishes
    const size_t rows = size_t(a.F) * a.ostride;
#pragma unroll
    for (int j = 0; j < MC; ++j) {
      const uint32_t m = mt * MT + (wm * MC + j) * 32u + fr;
      if (m >= a.M) continue;
#pragma unroll
      for (int i = 0; i < FC; ++i) {
        const uint32_t fb0 = f0 + (wf * FC + i) * 32u + 4u * (lane >> 5);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const uint32_t f = fb0 + 8u * uint32_t(v >> 2) + uint32_t(v & 3);
          if (f < a.F) a.part[(size_t(sp) * rows + size_t(f) * a.ostride + phase) * a.M + m] = acc[i][j][v];
        }
      }
    }
    return;
  }
  // epilogue: acc[i][j][v] = D[frame 8 (v/4) + 4 (lane/32) + v%4][channel lane%32].
  // Frames past F are stored like the others: they land behind the buffers'
  // last frame, in their tails.  Every address is a wave-uniform pointer plus
  // a lane offset that does not change from value to value.
  const uint32_t hl = lane >> 5, cc = fr >> 3, ts = a.M * 16u;  // ts: halfs between 16-frame tiles
  uint32_t lo[4];  // lane offsets in a plane, by the kinds of rows that a value index can have
#pragma unroll
  for (uint32_t e = 0; e < 4; ++e) {
    uint32_t row, chunk;
    if constexpr (OS == 1) {
      row = 4u * hl * 32u;
      chunk = cc ^ (2u * hl) ^ e;  // e: (v % 4 / 2) ^ (v / 4 % 2)
    } else if constexpr (OS == 2) {
      row = (8u * hl + phase) * 32u;
      chunk = cc ^ e ^ hl;
    } else if constexpr (OS == 4) {
      row = hl * ts + phase * 32u;
      chunk = cc ^ ((2u * e + (phase >> 1)) & 3u) ^ (e >> 1);
    } else {
      row = 2u * hl * ts + phase * 32u;
      chunk = cc ^ ((phase >> 1) & 3u) ^ e;  // e: v % 2
    }
    lo[e] = row + (chunk << 3) + (fr & 7u);
  }
  const uint32_t lres = 4u * hl * OS * a.ldres + fr, ly = 4u * hl * OS * a.ldy + fr;
  // The residual values of the next fragment are loaded before this one's
  // stores (the residual may be the output buffer itself; a value is read and
  // written by the same lane, before the stores of any later fragment).
  float rv[2][16];
  auto load_res = [&](float (&r)[16], int q) {
    const float* p = a.res + (size_t(f0 + (wf * FC + q % FC) * 32u) * OS + phase) * a.ldres + mt * MT + (wm * MC + q / FC) * 32u;
#pragma unroll
    for (int v = 0; v < 16; ++v) r[v] = p[size_t(8 * (v >> 2) + (v & 3)) * OS * a.ldres + lres];
  };
  if (a.res) load_res(rv[0], 0);
#pragma unroll
  for (int q = 0; q < MC * FC; ++q) {
    const int j = q / FC, i = q % FC;
    if (a.res && q + 1 < MC * FC) load_res(rv[(q + 1) & 1], q + 1);
    const uint32_t mb = mt * MT + (wm * MC + j) * 32u, m = mb + fr, fb0 = f0 + (wf * FC + i) * 32u;
    const float bias = a.bias[m];
    const float gam = a.gamma ? a.gamma[m] : 1.0f;
    const float alp = a.alpha ? snake_guard(a.alpha[m]) : 1.0f, inv = 1.0f / alp;
    float* y32 = a.y32 + (size_t(fb0) * OS + phase) * a.ldy + mb;
    const size_t hb = size_t(fb0 / 16u * OS) * ts + (mb >> 5) * 512u;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const uint32_t Q = v >> 2, e = v & 3;
      float val = __fadd_rn(acc[i][j][v], bias);
      if (a.gelu) val = gelu_as(val);
      if (a.gamma) val = __fmul_rn(val, gam);
      if (a.res) val = __fadd_rn(rv[q & 1][v], val);
      if (a.y32) (y32 + size_t(8 * Q + e) * OS * a.ldy)[ly] = val;
      if (a.alpha) val = snake(val, alp, inv);
      if (a.yh) {
        const _Float16 h = _Float16(val);
        const uint32_t kind = OS == 1 ? (e >> 1) ^ (Q & 1u) : OS == 8 ? (e & 1u) : e;
        const uint32_t k = OS == 1   ? (Q >> 1) * ts + (8u * (Q & 1u) + e) * 32u
                           : OS == 2 ? Q * ts + 2u * e * 32u
                           : OS == 4 ? 2u * Q * ts + 4u * e * 32u
                                     : (4u * Q + (e >> 1)) * ts + 8u * (e & 1u) * 32u;
        (a.yh + hb + k)[lo[kind]] = h;
        if (a.yl) (a.yl + hb + k)[lo[kind]] = _Float16(__fsub_rn(val, float(h)));
      }
      if (v % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Sum of the K splits (in split order) and the conv epilogue, one thread per
// output element (row, m), rows = F * ostride.
__global__ __launch_bounds__(256) void conv_split_reduce_kernel(ConvGemmArgs a, uint32_t splits) {
  const size_t rows = size_t(a.F) * a.ostride;
  const size_t idx = size_t(blockIdx.x) * 256u + threadIdx.x;
  if (idx >= rows * a.M) return;
  const size_t row = idx / a.M;
  const uint32_t m = uint32_t(idx - row * a.M);
  float acc = a.part[idx];
  for (uint32_t z = 1; z < splits; ++z) acc = __fadd_rn(acc, a.part[size_t(z) * rows * a.M + idx]);
  float val = __fadd_rn(acc, a.bias[m]);
  if (a.gelu) val = gelu_as(val);
  if (a.gamma) val = __fmul_rn(val, a.gamma[m]);
  if (a.res) val = __fadd_rn(a.res[row * a.ldres + m], val);
  if (a.y32) a.y32[row * a.ldy + m] = val;
  if (a.alpha) {
    const float alp = snake_guard(a.alpha[m]);
    val = snake(val, alp, 1.0f / alp);
  }
  if (a.yh) {
    const _Float16 h = _Float16(val);
    const size_t o = act_off(uint32_t(row), m, a.M);
    a.yh[o] = h;
    if (a.yl) a.yl[o] = _Float16(__fsub_rn(val, float(h)));
  }
}

// rvq_lookup_codes (codec.rs:2536-2596): one block per frame, 4 outputs per
// thread; every sum in the reference's order (bit-exact).
__global__ __launch_bounds__(256) void codec_rvq_kernel(RvqArgs a) {
  const uint32_t f = blockIdx.x;
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t o = threadIdx.x + 256u * k;
    float acc = 0.0f;
    for (uint32_t q = 0; q < 10; ++q) {
      int32_t code = a.codes[size_t(q) * a.F + f];
      if (code < 0 || uint32_t(code) >= a.cb_size[q]) {
        if (a.err) *a.err = 1u;
        code = 0;
      }
      const float* z = a.cb[q] + size_t(code) * 8u;
      const float* w = a.pw[q] + size_t(o) * 8u;
      float d = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) d = __fadd_rn(d, __fmul_rn(z[j], w[j]));
      acc = __fadd_rn(acc, __fadd_rn(d, a.pb[q][o]));
    }
    a.out[size_t(f) * 1024u + o] = acc;
  }
}

__global__ __launch_bounds__(256) void codec_check_codes_kernel(const int32_t* codes, uint32_t F, uint32_t* err) {
  const size_t i = size_t(blockIdx.x) * 256u + threadIdx.x;
  if (i >= size_t(10) * F) return;
  const int32_t c = codes[i];
  const int32_t size = i < F ? 4096 : 1024;
  if (c < 0 || c >= size) *err = 1u;
}

// apply_rope_normal (attention.rs:172-206) on four values of a head: pairs
// (x0, x1) -> (x0 c - x1 s, x0 s + x1 c) with the table's (cos, sin).
__device__ __forceinline__ float4 rope4(float4 x, const float2* cs) {
  const float4 t = *reinterpret_cast<const float4*>(cs);  // c0, s0, c1, s1
  return make_float4(__fsub_rn(__fmul_rn(x.x, t.x), __fmul_rn(x.y, t.y)),
                     __fadd_rn(__fmul_rn(x.x, t.y), __fmul_rn(x.y, t.x)),
                     __fsub_rn(__fmul_rn(x.z, t.z), __fmul_rn(x.w, t.w)),
                     __fadd_rn(__fmul_rn(x.z, t.w), __fmul_rn(x.w, t.z)));
}

// Windowed causal attention of the post-module transformer
// (forward_codec_transformer_layer_with_window, codec.rs:3278-3300, over
// gqa_decode_attention, attention.rs:208-247): block = 16 queries x one head,
// the 143 keys / values those queries see ([q0 - 127, q0 + 15]) staged in LDS,
// q and k turned by RoPE as they are
// (key rows padded to 68 floats: 16-byte aligned, and a 16-lane phase of
// float4 reads covers all 64 banks).  A wave takes 4 queries: lane j scores
// keys j and j + 64 of the query's window (four partial sums per dot
// product), softmax over the wave, the probabilities go through wave-private
// LDS, and lane d sums p_k v_k[d] (four partial sums).
constexpr uint32_t CA_Q = 16, CA_W = 128, CA_K = CA_Q + CA_W - 1, CA_KS = 68;
__global__ __launch_bounds__(256) void codec_attn_kernel(const float* qkv, uint32_t T, const float2* table,
                                                         float* out) {
  __shared__ __align__(16) float ks[CA_K * CA_KS];
  __shared__ __align__(16) float vs[CA_K * 64];
  __shared__ __align__(16) float qs[CA_Q * 64];
  __shared__ __align__(16) float ps[4][128];
  const uint32_t q0 = blockIdx.x * CA_Q, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t kstart = q0 >= CA_W - 1 ? q0 - (CA_W - 1) : 0u;
  const uint32_t kend = min(T, q0 + CA_Q);
  const uint32_t nk = kend - kstart;
  for (uint32_t e = tid; e < nk * 16u; e += 256u) {
    const uint32_t r = e >> 4, d4 = (e & 15u) * 4u;
    const float* src = qkv + size_t(kstart + r) * 3072u + h * 64u + d4;
    *reinterpret_cast<float4*>(ks + r * CA_KS + d4) =
        rope4(*reinterpret_cast<const float4*>(src + 1024), table + size_t(kstart + r) * 32u + d4 / 2u);
    *reinterpret_cast<float4*>(vs + r * 64u + d4) = *reinterpret_cast<const float4*>(src + 2048);
  }
  {
    const uint32_t r = tid >> 4, d4 = (tid & 15u) * 4u;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (q0 + r < T)
      v = rope4(*reinterpret_cast<const float4*>(qkv + size_t(q0 + r) * 3072u + h * 64u + d4),
                table + size_t(q0 + r) * 32u + d4 / 2u);
    *reinterpret_cast<float4*>(qs + r * 64u + d4) = v;
  }
  __syncthreads();
  float* pw = ps[wave];
  for (uint32_t qq = 0; qq < 4; ++qq) {
    const uint32_t ql = wave * 4u + qq, tq = q0 + ql;
    if (tq >= T) break;
    const uint32_t lo = tq >= CA_W - 1 ? tq - (CA_W - 1) : 0u, n = tq - lo + 1u;
    const float* qr = qs + ql * 64u;
    float sc[2];
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      const uint32_t j = lane + 64u * uint32_t(h2);
      sc[h2] = -INFINITY;
      if (j < n) {
        const float* kr = ks + (lo + j - kstart) * CA_KS;
        float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
        for (int i = 0; i < 64; i += 4) {
          const float4 qv = *reinterpret_cast<const float4*>(qr + i);
          const float4 kv = *reinterpret_cast<const float4*>(kr + i);
          a0 = fmaf(qv.x, kv.x, a0);
          a1 = fmaf(qv.y, kv.y, a1);
          a2 = fmaf(qv.z, kv.z, a2);
          a3 = fmaf(qv.w, kv.w, a3);
        }
        sc[h2] = ((a0 + a1) + (a2 + a3)) * 0.125f;
      }
    }
    const float mx = wave_max(fmaxf(sc[0], sc[1]));
    const float e0 = lane < n ? expf_glibc(sc[0] - mx) : 0.0f;
    const float e1 = lane + 64u < n ? expf_glibc(sc[1] - mx) : 0.0f;
    const float sum = wave_sum(e0 + e1);
    const float inv = 1.0f / sum;
    pw[lane] = e0 * inv;
    pw[lane + 64u] = e1 * inv;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float* vb = vs + (lo - kstart) * 64u + lane;
    float o0 = 0.f, o1 = 0.f, o2 = 0.f, o3 = 0.f;
    uint32_t k = 0;
    for (; k + 4u <= n; k += 4u) {
      const float4 p4 = *reinterpret_cast<const float4*>(pw + k);
      o0 = fmaf(p4.x, vb[(k + 0u) * 64u], o0);
      o1 = fmaf(p4.y, vb[(k + 1u) * 64u], o1);
      o2 = fmaf(p4.z, vb[(k + 2u) * 64u], o2);
      o3 = fmaf(p4.w, vb[(k + 3u) * 64u], o3);
    }
    for (; k < n; ++k) o0 = fmaf(pw[k], vb[k * 64u], o0);
    out[size_t(tq) * 1024u + h * 64u + lane] = (o0 + o1) + (o2 + o3);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

__global__ __launch_bounds__(256) void codec_split16_kernel(const float* x, _Float16* hi, _Float16* lo, size_t n,
                                                            uint32_t C) {
  const size_t i = size_t(blockIdx.x) * 256u + threadIdx.x;
  if (i >= n) return;
  const float v = x[i];
  const _Float16 h = _Float16(v);
  const size_t o = act_off(uint32_t(i / C), uint32_t(i % C), C);
  hi[o] = h;
  if (lo) lo[o] = _Float16(__fsub_rn(v, float(h)));
}

// forward_codec_convnext_block front (codec.rs:3444-3460): depthwise causal
// conv k7 (depthwise_causal_conv1d :3576-3619, sums in the reference order)
// then layer_norm_affine_frame_major (:3621-3654) over the frame's 1024
// channels; output as hi / lo planes for the pointwise product.
__global__ __launch_bounds__(256) void codec_dwconv_ln_kernel(const float* x, uint32_t F, const float* w,
                                                              const float* b, const float* ln_w, const float* ln_b,
                                                              float eps, _Float16* hi, _Float16* lo) {
  __shared__ float red[4];
  const uint32_t f = blockIdx.x, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  float d[4];
  float s = 0.0f;
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t c = tid + 256u * k;
    float acc = b[c];
#pragma unroll
    for (uint32_t kk = 0; kk < 7; ++kk) {
      if (f + kk < 6u) continue;
      const uint32_t src = f + kk - 6u;
      acc = __fadd_rn(acc, __fmul_rn(x[size_t(src) * 1024u + c], w[c * 7u + kk]));
    }
    d[k] = acc;
    s += acc;
  }
  s = wave_sum(s);
  if (lane == 0) red[wave] = s;
  __syncthreads();
  const float mean = ((red[0] + red[1]) + (red[2] + red[3])) / 1024.0f;
  __syncthreads();
  float v = 0.0f;
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const float c = d[k] - mean;
    v += c * c;
  }
  v = wave_sum(v);
  if (lane == 0) red[wave] = v;
  __syncthreads();
  const float var = ((red[0] + red[1]) + (red[2] + red[3])) / 1024.0f;
  const float scale = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(var, eps)));
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t c = tid + 256u * k;
    const float y = __fadd_rn(__fmul_rn(__fmul_rn(__fsub_rn(d[k], mean), scale), ln_w[c]), ln_b[c]);
    const _Float16 h = _Float16(y);
    const size_t o = act_off(f, c, 1024u);
    hi[o] = h;
    lo[o] = _Float16(__fsub_rn(y, float(h)));
  }
}

// Output conv of the decoder (96 -> 1, k 7, causal; causal_conv_1d_frame_major
// :2212-2293, sum = bias, then tap, then channel, in order) over the f16
// snake outputs, then tanh.  Block = 256 samples; the 262 input rows it reads
// are staged in LDS (row stride 98 halfs: 49 dwords, odd, so lanes reading
// consecutive rows hit distinct banks).
constexpr uint32_t OC_ROW = 98;
__global__ __launch_bounds__(256) void codec_out_conv_kernel(const _Float16* x, uint32_t T, const float* w, float b,
                                                             float* out) {
  __shared__ _Float16 xs[262 * OC_ROW];
  __shared__ float wsm[7][96];
  const uint32_t t0 = blockIdx.x * 256u, tid = threadIdx.x;
  for (uint32_t e = tid; e < 96u * 7u; e += 256u) wsm[e % 7u][e / 7u] = w[e];  // w[c][tap]
  for (uint32_t e = tid; e < 262u * 12u; e += 256u) {
    const uint32_t r = e / 12u, c = e - r * 12u;
    const int32_t src = int32_t(t0) + int32_t(r) - 6;
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (src >= 0 && src < int32_t(T)) v = *reinterpret_cast<const uint4*>(x + act_off(uint32_t(src), c * 8u, 96u));
    uint32_t* d = reinterpret_cast<uint32_t*>(xs + r * OC_ROW + c * 8u);
    d[0] = v.x;
    d[1] = v.y;
    d[2] = v.z;
    d[3] = v.w;
  }
  __syncthreads();
  const uint32_t t = t0 + tid;
  if (t >= T) return;
  float y = b;
  for (uint32_t tap = 0; tap < 7; ++tap) {
    const _Float16* row = xs + (tid + tap) * OC_ROW;
    for (uint32_t c = 0; c < 96; c += 2) {
      const uint32_t pr = *reinterpret_cast<const uint32_t*>(row + c);
      const float x0 = float(__builtin_bit_cast(_Float16, uint16_t(pr & 0xffffu)));
      const float x1 = float(__builtin_bit_cast(_Float16, uint16_t(pr >> 16)));
      y = __fadd_rn(y, __fmul_rn(x0, wsm[tap][c]));
      y = __fadd_rn(y, __fmul_rn(x1, wsm[tap][c + 1]));
    }
  }
  out[t] = tanhf(y);
}

template <int G, int PL, int MC, int FC, int WMG, int NB, int NA, bool FU, int OS>
hipError_t conv_gemm_launch(const ConvGemmArgs& a, uint32_t phases, hipStream_t s) {
  constexpr uint32_t MT = 32 * MC * WMG, FT = 32 * FC * (4 / WMG), AT = FT / 16 + (G == 7 ? 4 : G == 1 ? 0 : 1);
  constexpr uint32_t lds = NB * MT * 64 + NA * PL * AT * 1024;
  static_assert(!FU || FT * MT * 2 <= lds, "the k1 conv's input must fit the stage buffers");
  const int32_t last = a.off0 + int32_t(a.G - 1) * a.ostep;
  const int32_t wbase = a.off0 < last ? a.off0 : last, wend = a.off0 < last ? last : a.off0;
  // window: frames f0 + wbase .. f0 + FT - 1 + wend, from the 16-frame tile that holds its first
  if (wend > 0 || wbase < -ACT_GUARD) return hipErrorInvalidValue;
  const int32_t tile0 = -((15 - wbase) / 16), shift = wbase - 16 * tile0;
  const uint32_t a_tiles = (uint32_t(shift + (wend - wbase)) + FT + 15u) / 16u;
  if (a_tiles > AT) return hipErrorInvalidValue;
  static std::atomic<uint64_t> devices{0};
  const hipError_t attr = allow_lds(reinterpret_cast<const void*>(&conv_gemm_kernel<G, PL, MC, FC, WMG, NB, NA, FU, OS>), lds, devices);
  if (attr != hipSuccess) return attr;
  const uint32_t m_tiles = (a.M + MT - 1) / MT, f_tiles = (a.F + FT - 1) / FT;
  // K split when the grid would leave CUs idle: each split keeps >= 2 stages
  const uint32_t nst = a.C / 32, blocks = m_tiles * f_tiles * phases;
  const size_t rows = size_t(a.F) * phases;
  uint32_t splits = 1;
  if (a.part && !FU) {
    while (splits < 8 && blocks * splits < 256u && nst / (2 * splits) >= 2 &&
           size_t(2 * splits) * rows * a.M <= a.part_cap)
      splits *= 2;
  }
  // frame-tile-major block order when the weights of every (phase, m tile)
  // fit in an XCD's L2 next to the streamed input windows
  const size_t wbytes = size_t(phases) * m_tiles * a.G * MT * a.C * sizeof(_Float16);
  const uint32_t fmajor = wbytes <= CG_FMAJOR_WEIGHT_BYTES ? 1u : 0u;
  conv_gemm_kernel<G, PL, MC, FC, WMG, NB, NA, FU, OS><<<dim3(m_tiles * f_tiles * phases, 1, splits), 256, lds, s>>>(
      a, m_tiles, f_tiles, tile0, a_tiles, shift + a.off0 - wbase, a.ostep, fmajor);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || splits == 1) return e;
  const size_t n = rows * a.M;
  conv_split_reduce_kernel<<<uint32_t((n + 255) / 256), 256, 0, s>>>(a, splits);
  return hipGetLastError();
}

// Frames per wave: 64, or 32 where those tiles would leave fewer than two
// blocks per CU (37 code frames, us: transposed convs 34 / 50 / 43 / 33 -> 29 /
// 38 / 41 / 24, residual units of blocks 3 and 4 52 / 39 -> 42 / 29).  Where the line
// lies, whole decodes in ms with 64 frames always : from 256 : from 512 : from 1024
// blocks : never: 37 code frames 1.94 : 1.84 : 1.77 : 1.77 : 1.77, 130 3.31 : 3.25 :
// 3.26 : 3.11 : 2.93, 180 3.62 : 3.51 : 3.52 : 3.47 : 3.45, 260 4.98 : 4.93 : 4.88 :
// 4.89 : 4.75, 350 5.75 : 5.68 : 5.67 : 5.69 : 5.72, 512 7.51 : 7.48 : 7.45 : 7.56 :
// 7.82 (block 3's transposed conv 376 -> 424 us).
template <int G, int PL, int MC, int WMG, int NB, int NA, bool FU, int OS>
hipError_t conv_gemm_frames(const ConvGemmArgs& a, uint32_t phases, hipStream_t s) {
  constexpr uint32_t MT = 32 * MC * WMG, FT = 64 * (4 / WMG);
  const uint32_t blocks = (a.M + MT - 1) / MT * ((a.F + FT - 1) / FT) * phases;
  if (blocks < 512u) return conv_gemm_launch<G, PL, MC, 1, WMG, NB, NA, FU, OS>(a, phases, s);
  return conv_gemm_launch<G, PL, MC, 2, WMG, NB, NA, FU, OS>(a, phases, s);
}

}  // namespace

uint32_t conv_tile_rows(uint32_t M) { return M % 192u == 0 ? 192u : M % 96u == 0 ? 96u : 256u; }

size_t conv_packed_halfs(uint32_t phases, uint32_t M, uint32_t G, uint32_t C) {
  const uint32_t MT = conv_tile_rows(M);
  return size_t(phases) * ((M + MT - 1) / MT) * MT * G * C;
}

hipError_t launch_conv_gemm(const ConvGemmArgs& a, uint32_t phases, hipStream_t s) {
  if (a.C == 0 || a.C % 32 || a.F == 0 || a.M == 0 || a.M % 32 || phases == 0) return hipErrorInvalidValue;
  if (uint64_t(a.F) * phases > 0x7fffffffull) return hipErrorInvalidValue;
  const bool split = a.xl != nullptr;
  const uint32_t MT = conv_tile_rows(a.M);
  if (a.M % MT || a.ostride != phases) return hipErrorInvalidValue;
  const uint32_t os = a.ostride;
  if (MT == 192 && a.G == 7 && !split && os == 1) return conv_gemm_frames<7, 1, 3, 2, 3, 2, false, 1>(a, phases, s);
  if (MT == 192 && a.G == 1 && !split && os == 1) return conv_gemm_frames<1, 1, 3, 2, 3, 3, false, 1>(a, phases, s);
  if (MT == 192 && a.G == 2 && split && os == 8) return conv_gemm_frames<2, 2, 3, 2, 3, 2, false, 8>(a, phases, s);
  if (MT == 192 && a.G == 2 && split && os == 4) return conv_gemm_frames<2, 2, 3, 2, 3, 2, false, 4>(a, phases, s);
  if (MT == 96 && a.G == 2 && split && os == 2) return conv_gemm_frames<2, 2, 3, 1, 2, 2, false, 2>(a, phases, s);
  if (MT == 256 && a.G == 1 && split && os == 2) return conv_gemm_frames<1, 2, 4, 2, 2, 2, false, 2>(a, phases, s);
  if (MT == 256 && a.G == 1 && split && os == 1) return conv_gemm_frames<1, 2, 4, 2, 2, 2, false, 1>(a, phases, s);
  return hipErrorInvalidValue;
}

bool residual_unit_fits(uint32_t M) { return M == 96 || M == 192; }

hipError_t launch_residual_unit(const ConvGemmArgs& a, hipStream_t s) {
  if (!a.w1 || !a.bias_mid || !a.alpha_mid || !residual_unit_fits(a.M) || a.G != 7 || a.xl || a.C != a.M || a.F == 0)
    return hipErrorInvalidValue;
  if (a.M == 192) return conv_gemm_frames<7, 1, 3, 2, 3, 2, true, 1>(a, 1, s);
  return conv_gemm_frames<7, 1, 3, 1, 4, 2, true, 1>(a, 1, s);
}

hipError_t launch_codec_rvq(const RvqArgs& a, hipStream_t s) {
  if (a.F == 0) return hipSuccess;
  codec_rvq_kernel<<<a.F, 256, 0, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_codec_check_codes(const int32_t* codes, uint32_t F, uint32_t* err, hipStream_t s) {
  const size_t n = size_t(10) * F;
  if (n == 0) return hipSuccess;
  codec_check_codes_kernel<<<uint32_t((n + 255) / 256), 256, 0, s>>>(codes, F, err);
  return hipGetLastError();
}

hipError_t launch_codec_attention(const float* qkv, uint32_t T, const float2* table, float* out, hipStream_t s) {
  if (T == 0) return hipSuccess;
  codec_attn_kernel<<<dim3((T + CA_Q - 1) / CA_Q, 16), 256, 0, s>>>(qkv, T, table, out);
  return hipGetLastError();
}

hipError_t launch_codec_split16(const float* x, _Float16* hi, _Float16* lo, size_t frames, uint32_t C, hipStream_t s) {
  const size_t n = frames * C;
  if (n == 0) return hipSuccess;
  codec_split16_kernel<<<uint32_t((n + 255) / 256), 256, 0, s>>>(x, hi, lo, n, C);
  return hipGetLastError();
}

hipError_t launch_codec_dwconv_ln(const float* x, uint32_t F, const float* w, const float* b, const float* ln_w,
                                  const float* ln_b, float eps, _Float16* hi, _Float16* lo, hipStream_t s) {
  if (F == 0) return hipSuccess;
  codec_dwconv_ln_kernel<<<F, 256, 0, s>>>(x, F, w, b, ln_w, ln_b, eps, hi, lo);
  return hipGetLastError();
}

hipError_t launch_codec_out_conv(const _Float16* x, uint32_t T, const float* w, float b, float* out, hipStream_t s) {
  if (T == 0) return hipSuccess;
  codec_out_conv_kernel<<<(T + 255) / 256, 256, 0, s>>>(x, T, w, b, out);
  return hipGetLastError();
}

}  // namespace s2
