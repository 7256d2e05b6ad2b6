// Whisper encoder kernels for gfx950: an MFMA GEMM with fused epilogues (also used as an
// implicit-GEMM conv1d and for the decoder cross K/V projection) and a row LayerNorm; the encoder
// self-attention is in attention_enc.hip. Semantics follow HF WhisperEncoder.forward in fp16
// (transformers models/whisper/modeling_whisper.py:592-648, layer :379-414, attention :284-358):
// every op output is rounded to fp16, accumulation is fp32.
#include <type_traits>

#include "lds_pipe.h"

namespace fw {
namespace {

// ------------------------------------------------------------------------------------------
// GEMM: out[m, n] = epi(sum_k A[m, k] * W[n, k]).  Block tile BM x 128 x 64 with BM in
// {256, 192, 128, 64}; waves in a (BM / 64 or 2) x 2 arrangement, each wave a (64 or 32) x 64 tile of
// v_mfma_f32_32x32x16_f16 products (192-row tiles: 2 x 4 waves of 96 x 32; 64-row tiles: 2 x 4 waves
// of 32 x 32).
//  - LDS: one [rows][64] fp16 tile per operand and stage, 8 x 16-byte chunks per row, chunk c of
//    row r stored in slot swz_slot(r, c) = c ^ ((r >> 1) & 7), so the 16 rows a 16-lane group reads
//    for one MFMA operand cover all 64 banks (conflict-free ds_read_b128).
//  - Epilogues: bias, GELU (erfc by a fitted exponent polynomial, one fp16 ulp of the exact-erf GELU at most),
//    residual, fp16 clamp, the q scale, the cross K/V scatter and the transposed-V store.
//  - Plain GEMMs (gemm_dma_kernel): global -> LDS copies into a ring of stages, operand fragments
//    double-buffered in registers (see the pipeline notes above that kernel).
//  - Implicit-GEMM conv: a 64-wide k stage of A row m is 64 contiguous channels of input row
//    m * stride + tap - 1, so convs use the same direct-to-LDS pipeline, from a raw buffer whose range check
//    gives the padding rows' zeros (inputs of 2 GiB and more: 64-bit addresses, padding from a zero row).
//  - Products of few rows: tiles of 32 x 32 to 64 x 64 (split products: 96 x 64) whose k stages are dealt to
//    the block's waves (gemm_ks_kernel); choose_tile picks the tile by the passes over the CUs and their cost.
//  - Tile order: hardware deals blocks round-robin over the 8 XCDs; the block id is remapped so each
//    XCD works on its own part of the tile grid and its L2 sees only that part's operand panels.
// MFMA 32x32x16 f16 operand layout (lane l, g = l / 32):
//   A: lane holds A[l % 32][8g .. 8g + 7]      B: lane holds B[8g .. 8g + 7][l % 32]
//   C: acc[r] = C[8 (r / 4) + 4 g + (r % 4)][l % 32], r = 0 .. 15
// ------------------------------------------------------------------------------------------
constexpr int kBN = 128, kBK = 64;
constexpr int kEpiCrossKV = 100;  // internal epilogue: scatter into [layers, 2, heads, t, 64]
// Internal epilogue of the encoder q/k/v projection: q columns scaled as FW_EPI_SCALE_Q, k columns
// stored as they are, v columns stored transposed into vt (the attention kernel's V layout).
constexpr int kEpiQkvVt = 101;
// Internal epilogue of the split-k products: split s (blockIdx.x / tiles) covers k in [s k, (s + 1) k)
// and stores its fp32 sums to part[s][m][n]; the row kernel that follows adds the splits.
constexpr int kEpiPartial = 102;

struct GemmArgs {
  const _Float16* a;
  int lda;
  const _Float16* w;
  int ldw;
  const _Float16* bias;
  _Float16* out;
  int ldo;
  const _Float16* res;
  int ldr;
  int m, n, k;
  int q_cols;
  // implicit conv1d (k = 3, pad 1): a is x[t_in, c_in]; row m, column kk = tap * c_in + c reads
  // x[m * stride + tap - 1, c], zero outside [0, t_in).
  int conv_stride;  // 0: plain GEMM
  int t_in, c_in;
  // cross K/V scatter
  int heads, t_len;
  // q/k/v projection: transposed V, [heads * 64][vt_pad]
  _Float16* vt;
  int vt_pad;
  // XCD tile grouping (0: none): the 8 XCDs split the tile grid into xm x xn rectangles
  int xm, xn;
  // split-k products (kEpiPartial): number of splits and the fp32 partial sums [splits][m][n]
  int splits;
  float* part;
};

// The first 14 dwords of a kernel's arguments arrive in scalar registers with the launch (the build preloads
// them); the rest is a read of the argument segment, a memory round trip at the head of every launch.
// So what the first copies need comes as arguments of its own, ahead of the struct (the encoder of a full
// window 4040 -> 3951 us, over 251 frames, 4 layers, 311 -> 294 us).
#define FW_GEMM_PARAMS                                                                                       \
  const _Float16 *a_, const _Float16 *w_, int lda_, int ldw_, int m_, int n_, int k_, int splits_, int xcd_, \
      int conv_stride_, int t_in_, int c_in_, GemmArgs g
#define FW_GEMM_ARGS(g) \
  g.a, g.w, g.lda, g.ldw, g.m, g.n, g.k, g.splits, g.xm | g.xn << 8, g.conv_stride, g.t_in, g.c_in, g
#define FW_GEMM_TAKE_PARAMS()                                                        \
  g.a = a_, g.w = w_, g.lda = lda_, g.ldw = ldw_, g.m = m_, g.n = n_, g.k = k_,      \
  g.splits = splits_, g.xm = xcd_ & 255, g.xn = xcd_ >> 8, g.conv_stride = conv_stride_, g.t_in = t_in_, g.c_in = c_in_

// Block -> output tile. Hardware deals workgroups round-robin over the 8 XCDs (block b runs on XCD
// b % 8), each with its own L2. With a grouping, XCD x owns one (ntm / xm) x (ntn / xn) rectangle of
// the tile grid, so each XCD fetches only its slices of A and W. Otherwise each XCD takes a contiguous
// run of row-major tiles (the tail beyond a multiple of 8 keeps its id). Both maps are bijective.
template <int BM, int BN = kBN>
__device__ __forceinline__ void tile_origin(const GemmArgs& g, int& m0, int& n0) {
  const int ntn = g.n / BN, ntm = (g.m + BM - 1) / BM;
  const int bid = g.splits > 1 ? static_cast<int>(blockIdx.x) % (ntn * ntm) : static_cast<int>(blockIdx.x);
  int tm, tn;
  if (g.xm) {
    const int xcd = bid & 7, local = bid >> 3, mr = ntm / g.xm, nr = ntn / g.xn;
    tm = (xcd / g.xn) * mr + local % mr;
    tn = (xcd % g.xn) * nr + local / mr;
  } else {
    const int ntiles = ntn * ntm, full = (ntiles / 8) * 8;
    const int tile = bid < full ? (bid % 8) * (full / 8) + bid / 8 : bid;
    tm = tile / ntn;
    tn = tile % ntn;
  }
  m0 = tm * BM;
  n0 = tn * BN;
}

constexpr bool epi_reads_res(int epi) {
  return epi == FW_EPI_BIAS_RESID || epi == FW_EPI_BIAS_RESID_CLAMP || epi == FW_EPI_BIAS_GELU_POS;
}

// GELU(x) = x Phi(x) with Phi(x) = erfc(-x / sqrt 2) / 2, written as in Press et al., Numerical
// Recipes in C (2nd ed.), 6.2 ("erfcc"): with z = |x| / sqrt 2 and t = 1 / (1 + z / 2),
//   erfc(z) / 2 = t 2^(Q(t) - z^2 log2 e),
// where Q(t) = log2(erfc(z) / (2 t)) + z^2 log2 e is smooth in t. Q here is our own degree-7 fit
// (near-minimax by iteratively reweighted least squares against float64 erfc on t in [0.3, 1], i.e.
// z <= 4.67; max |error| 4.0e-7 in log2 units, so erfc carries a relative error below 3e-7), with the
// 1/2 and the log2 e scaling folded into the coefficients. On both tails the result is accurate in
// relative terms; rounded to fp16 it equals the exact-erf GELU on all but 7 of the finite fp16
// inputs, which are one ulp off (the same count as the Numerical Recipes coefficients, which cost
// two more FMAs and three more scalings per element; the fc1 epilogue is bound by VALU issue).
// Beyond z = 4.67 the GELU underflows fp16 on the negative side and equals x on the positive side.
// The product x Phi(x) is rounded once, to fp16 (v_fma_mixlo_f16; issued as assembly, because whether the
// compiler picks it or an fp32 product and a conversion, which rounds twice, depends on what stands around it).
__device__ __forceinline__ _Float16 gelu_enc(_Float16 xh) {
  const float x = h2f(xh);
  const float t = __builtin_amdgcn_rcpf(fmaf(fabsf(x), 0.35355339059327376f, 1.0f));
  float q = -0.19670111f;
  q = fmaf(t, q, 0.74583995f);
  q = fmaf(t, q, -0.79930210f);
  q = fmaf(t, q, -0.15935127f);
  q = fmaf(t, q, 0.34100536f);
  q = fmaf(t, q, 0.42959806f);
  q = fmaf(t, q, 1.46661794f);
  q = fmaf(t, q, -2.82770705f);
  const float c = t * __builtin_amdgcn_exp2f(fmaf(x * x, -0.72134752f, q));  // Phi(-|x|)
  const float phi = x >= 0.0f ? 1.0f - c : c;
  _Float16 y;
  asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "=v"(y) : "v"(phi), "v"(xh));
  return y;
}

// The epilogue's value before its residual / position operand: an fp16 number for the epilogues that read
// one, so it can be staged as fp16 without a rounding of its own.
template <int EPI>
__device__ __forceinline__ float epilogue_pre(float acc, float b, int col, int q_cols) {
  if constexpr (EPI == FW_EPI_BIAS_GELU || EPI == FW_EPI_BIAS_GELU_POS) return h2f(gelu_enc(f2h(acc + b)));
  float v = round_h(acc + b);
  if constexpr (EPI == FW_EPI_SCALE_Q || EPI == kEpiQkvVt)
    if (col < q_cols) v = v * 0.125f;
  return v;
}
// The value before the final fp16 rounding, from epilogue_pre's and the operand.
template <int EPI>
__device__ __forceinline__ float epilogue_res(float v, float res) {
  v = res + v;
  if constexpr (EPI == FW_EPI_BIAS_RESID_CLAMP) {
    const float c = 65504.0f - 1000.0f;
    v = fminf(fmaxf(round_h(v), -c), c);
  }
  return v;
}

// Rows of fp16 outputs and operands are moved 16 bytes at a time whatever their alignment (the hardware
// takes unaligned global accesses; the encoder's own are aligned).
typedef _Float16 h8u __attribute__((ext_vector_type(8), aligned(2)));
typedef _Float16 h4u __attribute__((ext_vector_type(4), aligned(2)));

// MFMA operand fragments of one 64-wide k stage for a wave: A rows wm + 32 i + lane % 32, B rows
// wn + 32 j + lane % 32, k-step s covering k 16 s .. 16 s + 15.
template <int kTM, int kTN>
struct Frags {
  h8v a[kBK / 16][kTM];
  h8v b[kBK / 16][kTN];
};

// Byte offsets, within one ring stage (A tile, then the B tile at BM * 128 bytes), of a lane's
// fragments for each k-step s. Rows wm + 32 i + lr and wm + lr have the same swizzle (wm and 32 i are
// multiples of 16), so row group i (or j) is the k-step's offset plus 4096 i bytes, an immediate of
// the LDS read: a stage's reads then cost one address add per k-step and operand.
struct FragOffsets {
  uint32_t a[kBK / 16], b[kBK / 16];
};
static_assert(FW_SWZ_SHIFT <= 2, "fragment offsets need rows r and r + 32 to share the swizzle");

template <int BM>
__device__ __forceinline__ FragOffsets frag_offsets(int wm, int wn, int lr, int lg) {
  FragOffsets o;
#pragma unroll
  for (int s = 0; s < kBK / 16; ++s) {
    o.a[s] = static_cast<uint32_t>(swz(wm + lr, 2 * s + lg) * 16);
    o.b[s] = static_cast<uint32_t>(BM * 128 + swz(wn + lr, 2 * s + lg) * 16);
  }
  return o;
}

template <int kTM, int kTN>
__device__ __forceinline__ void load_frags(const char* stage, const FragOffsets& o, Frags<kTM, kTN>& f) {
#pragma unroll
  for (int s = 0; s < kBK / 16; ++s) {
#pragma unroll
    for (int i = 0; i < kTM; ++i) f.a[s][i] = *reinterpret_cast<const h8v*>(stage + o.a[s] + 4096 * i);
#pragma unroll
    for (int j = 0; j < kTN; ++j) f.b[s][j] = *reinterpret_cast<const h8v*>(stage + o.b[s] + 4096 * j);
  }
}

// kT: accumulate the transposed tile (W rows as the MFMA A operand), so that acc[i][j][r] holds
// C[32 i + lane % 32][32 j + 8 (r / 4) + 4 g + r % 4]: four adjacent output columns per lane, which
// the epilogue stages as one 8-byte (fp32 sums: 16-byte) LDS access.
template <int kTM, int kTN, bool kT>
__device__ __forceinline__ void mma_frags(const Frags<kTM, kTN>& f, f16v (&acc)[kTM][kTN]) {
#pragma unroll
  for (int s = 0; s < kBK / 16; ++s)
#pragma unroll
    for (int i = 0; i < kTM; ++i)
#pragma unroll
      for (int j = 0; j < kTN; ++j) {
        if constexpr (kT)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.b[s][j], f.a[s][i], acc[i][j], 0, 0, 0);
        else
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[s][i], f.b[s][j], acc[i][j], 0, 0, 0);
      }
}

// ---- direct-to-LDS pipeline (plain GEMMs) ------------------------------------------------------
// Per stage kt: wait until stage kt + 1 has landed, barrier (every wave also holds stage kt's operand
// fragments in registers by then, so its LDS slot is free), refill that slot with stage kt + ST,
// start the LDS reads of stage kt + 1's fragments, and run stage kt's MFMAs while they arrive. Copies
// have ST - 1 stages of MFMA time to land and LDS read latency is hidden behind the MFMAs.
// The LDS ring depth ST is picked per tile height: 256-row tiles use three 48 KB stages (one 8-wave
// block per CU); 128-row tiles (8 waves of 32 x 64; the split-k products) four 32 KB stages; 64-row
// tiles (launched when 128-row tiles would leave CUs idle) four 24 KB stages (5 or 6 measured the same).
// Tuning knobs (defaults measured on MI355X): ring depths per tile height, waves per 256-row and 64-row
// block, and the XCD rectangle grouping.
// 8 waves on the 64-row tiles (two per SIMD) against 4: out projection 14.8 -> 14.35 us, stem conv
// 36.0 -> 33.0 us (kernel trace, same box).
#ifndef FW_ST128
#define FW_ST128 4
#endif
#ifndef FW_ST64
#define FW_ST64 4
#endif
#ifndef FW_ST256
#define FW_ST256 3
#endif
#ifndef FW_ST192
#define FW_ST192 3
#endif
template <int BM>
constexpr int dma_stages() {
  return BM == 256 ? FW_ST256 : BM == 192 ? FW_ST192 : BM == 128 ? FW_ST128 : FW_ST64;
}
// Ring depths: at least two stages (one read while the next lands) and a ring that fits the 160 KB of
// LDS of a CU; the vmcnt range of the explicit waits is checked where they are instantiated.
template <int BM>
constexpr bool ring_fits() { return dma_stages<BM>() >= 2 && dma_stages<BM>() * (BM + kBN) * 128 <= 160 * 1024; }
static_assert(ring_fits<256>() && ring_fits<192>() && ring_fits<128>() && ring_fits<64>(),
              "FW_ST256 / FW_ST192 / FW_ST128 / FW_ST64: 2 or more stages within 160 KB of LDS");
// Waves per block, in gemm_wave_cols columns (kBN / cols output columns each) and waves / cols rows;
// each wave owns a (BM / rows) x (kBN / cols) tile. 192-row tiles use 2 x 4 waves of 96 x 32 and
// 128-row tiles 4 x 2 waves of 32 x 64.
#ifndef FW_W256
#define FW_W256 8
#endif
static_assert(FW_W256 == 2 || FW_W256 == 4 || FW_W256 == 8 || FW_W256 == 16,
              "FW_W256: 2 x (FW_W256 / 2) waves, each a whole number of 32-row MFMA tiles of the 256 rows");
#ifndef FW_W64
#define FW_W64 8  // waves per 64-row block: 8 (2 x 4 of 32 x 32) or 4 (2 x 2 of 32 x 64)
#endif
static_assert(FW_W64 == 4 || FW_W64 == 8, "FW_W64: 4 or 8 waves per 64-row block");
template <int BM>
constexpr int gemm_waves() { return BM == 256 ? FW_W256 : BM == 192 || BM == 128 ? 8 : FW_W64; }
template <int BM>
constexpr int gemm_wave_cols() { return BM == 192 || (BM == 64 && FW_W64 == 8) ? 4 : 2; }

// Source of the implicit conv's zero padding rows: a k stage of one A row is 64 halves.
__device__ __align__(16) _Float16 g_zero_row[kBK];

// Implicit conv1d (k = 3, pad 1) of any size: a 64-wide k stage lies inside one tap (c_in % 64 == 0), so
// A row m of the stage is 64 contiguous channels of input row m * stride + tap - 1, or zeros outside
// [0, t_in).
template <int BM>
__device__ __forceinline__ void dma_stage_conv(const GemmArgs& g, int m0, int n0, int k0, int wave, int lane,
                                          uint32_t lds_stage) {
  constexpr int kAInstr = BM / 8 / gemm_waves<BM>();  // wave instructions per A tile (8 rows each), per wave
  constexpr int kBInstr = kBN / 8 / gemm_waves<BM>();
  const int rsub = lane >> 3, slot = lane & 7;
  const int tap = k0 / g.c_in, ch0 = k0 - tap * g.c_in;
#pragma unroll
  for (int i = 0; i < kAInstr; ++i) {
    const int blk = wave * kAInstr + i;  // 8-row block of the tile
    const int row = blk * 8 + rsub;
    const int gm = min(m0 + row, g.m - 1);  // rows past m are computed and never stored
    const int chunk = swz_slot(row, slot);
    const int r = gm * g.conv_stride + tap - 1;
    const _Float16* src =
        (r >= 0 && r < g.t_in) ? g.a + static_cast<size_t>(r) * g.c_in + ch0 + chunk * 8 : g_zero_row + chunk * 8;
    dma16(src, __builtin_amdgcn_readfirstlane(lds_stage + blk * 1024));
  }
#pragma unroll
  for (int i = 0; i < kBInstr; ++i) {
    const int blk = wave * kBInstr + i;
    const int row = blk * 8 + rsub;
    const int chunk = swz_slot(row, slot);
    dma16(g.w + static_cast<size_t>(n0 + row) * g.ldw + k0 + chunk * 8,
          __builtin_amdgcn_readfirstlane(lds_stage + BM * 128 + blk * 1024));
  }
}

// Plain GEMMs: the same copies with the k offset of a stage in the scalar base. Each lane keeps the
// byte offset of its 16-byte chunk (row * ld + swizzled chunk) for every copy it issues, so a stage
// costs kA + kB copy instructions and no vector address arithmetic (the per-stage 64-bit address
// updates were half the vector instructions of the main loop). The host keeps both operands below
// 4 GiB, the range of the 32-bit offsets.
template <int BM, int kNW>
struct CopyOffsets {
  static constexpr int kA = BM / 8 / kNW, kB = kBN / 8 / kNW;  // copies per wave and stage
  uint32_t a[kA], b[kB];
};

template <int BM, int kNW>
__device__ __forceinline__ void copy_offsets(const GemmArgs& g, int m0, int n0, int wave, int lane,
                                             CopyOffsets<BM, kNW>& c) {
  using C = CopyOffsets<BM, kNW>;
  const int rsub = lane >> 3, slot = lane & 7;
#pragma unroll
  for (int i = 0; i < C::kA; ++i) {
    const int row = (wave * C::kA + i) * 8 + rsub;
    const int gm = min(m0 + row, g.m - 1);  // rows past m are computed and never stored
    c.a[i] = static_cast<uint32_t>((static_cast<size_t>(gm) * g.lda + swz_slot(row, slot) * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < C::kB; ++i) {
    const int row = (wave * C::kB + i) * 8 + rsub;
    c.b[i] = static_cast<uint32_t>((static_cast<size_t>(n0 + row) * g.ldw + swz_slot(row, slot) * 8) * 2);
  }
}

// Implicit convs: row m, tap, channel ch of A is input row m * stride + tap - 1, that is x[m * stride *
// c_in - c_in + kk] at column kk = tap * c_in + ch. So A is a matrix of pitch stride * c_in that starts one
// input row early, and a copy's source is again a per-lane offset plus a scalar one. Only row 0 at the
// first tap and the last input row's successor at the third fall outside x: their lanes' offsets point past
// the buffer's end there, which reads as zero (3000 -> 1500 x 1280, k = 3840: 29.5 against 31.6 us with the
// source row worked out, compared and selected for every copy). Buffers of less than 2 GiB only. The scalar
// offset, up to the start of the third tap's last stage, is taken from the buffer's length before a lane's
// offset is compared, so the length is at least three rows: a one-row input would let it run past the end
// and the difference wrap. Every lane that reads outside x has the offset past the end, whatever the length.
__host__ __device__ constexpr int64_t conv_buffer_rows(int t_in) { return t_in + int64_t{1} > 3 ? t_in + int64_t{1} : 3; }
struct ConvSource {
  buffer_rsrc x;
  __device__ __forceinline__ explicit ConvSource(const GemmArgs& g)
      : x(make_rsrc(g.a - g.c_in, static_cast<uint32_t>(conv_buffer_rows(g.t_in) * g.c_in * 2))) {}
  // this lane's chunk of A row gm, LDS row `row`, slot `slot`: its offset at each tap
  __device__ __forceinline__ static void offsets(const GemmArgs& g, int gm, int row, int slot, uint32_t (&o)[3]) {
    const int r = gm * g.conv_stride;
    o[1] = static_cast<uint32_t>((r * g.c_in + swz_slot(row, slot) * 8) * 2);
    o[0] = r > 0 ? o[1] : kPastEnd;
    o[2] = r + 1 < g.t_in ? o[1] : kPastEnd;
  }
  __device__ __forceinline__ void copy(const uint32_t (&o)[3], int tap, uint32_t kk, uint32_t lds_base) const {
    dma16_buf(tap == 0 ? o[0] : tap == 1 ? o[1] : o[2], x, kk * 2, lds_base);
  }
};
bool conv_offsets_fit(const GemmArgs& g) { return conv_buffer_rows(g.t_in) * g.c_in * 2 < kPastEnd; }

template <int BM, int kNW>
__device__ __forceinline__ void dma_stage_w(const GemmArgs& g, const CopyOffsets<BM, kNW>& c, int kt, int wave,
                                            uint32_t lds_stage) {
  using C = CopyOffsets<BM, kNW>;
  const char* wb = reinterpret_cast<const char*>(g.w) + static_cast<size_t>(kt) * (kBK * 2);
#pragma unroll
  for (int i = 0; i < C::kB; ++i) dma16_s(c.b[i], wb, lds_stage + BM * 128 + (wave * C::kB + i) * 1024);
}

template <int BM, int kNW>
__device__ __forceinline__ void dma_stage_s(const GemmArgs& g, const CopyOffsets<BM, kNW>& c, int kt, int wave,
                                            uint32_t lds_stage) {
  using C = CopyOffsets<BM, kNW>;
  const char* ab = reinterpret_cast<const char*>(g.a) + static_cast<size_t>(kt) * (kBK * 2);
#pragma unroll
  for (int i = 0; i < C::kA; ++i) dma16_s(c.a[i], ab, lds_stage + (wave * C::kA + i) * 1024);
  dma_stage_w<BM, kNW>(g, c, kt, wave, lds_stage);
}

// v columns of the q/k/v projection -> vt[head * 64 + d][vt_pos(t)]; rows in [m, vt_pad) get zeros so
// the padding keys of the last attention tile hold finite values. The tile is transposed through LDS
// (the operand ring is free once every wave has left the main loop): each lane puts its 4-row runs
// into a [128 columns][BM] staging tile, already in vt_pos order (tiles start at multiples of 64 and
// vt_pos permutes within 16-key groups), and the block then writes each column's BM keys as whole
// 16-byte chunks instead of one 8-byte store per 4 keys and column.
template <int BM, int kTM, int kTN, int ST>
__device__ __forceinline__ void store_vt(const GemmArgs& g, const f16v (&acc)[kTM][kTN], int m0, int n0, int wm,
                                         int wn, int lr, int lg, u32x4* lds) {
  constexpr int kStride = BM + 8;  // halves per staged column (16-byte aligned rows)
  static_assert(kBN * kStride * 2 <= ST * (BM + kBN) * 128, "staging tile must fit the ring");
  _Float16* t = reinterpret_cast<_Float16*>(lds);
  __syncthreads();  // every wave has read its last operand fragments from the ring
#pragma unroll
  for (int j = 0; j < kTN; ++j) {
    const int cl = wn + 32 * j + lr;
    const float b = g.bias ? h2f(g.bias[n0 + cl]) : 0.f;
#pragma unroll
    for (int i = 0; i < kTM; ++i)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const int rl = wm + 32 * i + 8 * rq + 4 * lg;  // rows rl .. rl + 3 stay adjacent under vt_pos
        h4v v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = m0 + rl + e < g.m ? f2h(acc[i][j][4 * rq + e] + b) : static_cast<_Float16>(0.f);
        *reinterpret_cast<h4v*>(t + cl * kStride + vt_pos(rl)) = v;
      }
  }
  __syncthreads();
  constexpr int kChunks = BM / 8;  // 16-byte chunks per staged column
  _Float16* dst = g.vt + static_cast<size_t>(n0 - 2 * g.q_cols) * g.vt_pad;
  for (int c = threadIdx.x; c < kBN * kChunks; c += blockDim.x) {
    const int cl = c / kChunks, ch = c - cl * kChunks;
    const int pos = m0 + ch * 8;
    if (pos < g.vt_pad)
      *reinterpret_cast<u32x4*>(dst + static_cast<size_t>(cl) * g.vt_pad + pos) =
          *reinterpret_cast<const u32x4*>(t + cl * kStride + ch * 8);
  }
}

constexpr int kNoConv = 0, kConvBuffer = 1, kConvAny = 2;  // conv sources through a buffer, or worked out for any size

template <int BM, int EPI, int CONV = kNoConv, int ST = dma_stages<BM>()>
__global__ void __launch_bounds__(gemm_waves<BM>() * 64) gemm_dma_kernel(FW_GEMM_PARAMS) {
  FW_GEMM_TAKE_PARAMS();
  constexpr int kDmaStages = ST, kNW = gemm_waves<BM>(), kNWN = gemm_wave_cols<BM>();
  constexpr int kWM = BM / (kNW / kNWN), kTM = kWM / 32, kTN = kBN / kNWN / 32;
  static_assert(kWM % 32 == 0 && kTN >= 1 && BM % (8 * kNW) == 0, "wave tiling");
  constexpr int kStageBytes = (BM + kBN) * 128;
  constexpr int kPerStage = (BM / 8 / kNW) + (kBN / 8 / kNW);  // copies per thread per stage
  __shared__ __align__(1024) u32x4 lds[kDmaStages * kStageBytes / 16];

  int m0, n0;
  tile_origin<BM>(g, m0, n0);
  int split = 0;
  if constexpr (EPI == kEpiPartial) {  // this block's k range: [split k, (split + 1) k) of the rows
    split = static_cast<int>(blockIdx.x) / ((g.n / kBN) * ((g.m + BM - 1) / BM));
    g.a += static_cast<size_t>(split) * g.k;
    g.w += static_cast<size_t>(split) * g.k;
  }
  // wave is uniform: the copies' LDS targets and the offsets that depend on it stay scalar
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave / kNWN) * kWM, wn = (wave % kNWN) * (kBN / kNWN);
  const int lr = lane & 31, lg = lane >> 5;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const char* lds_bytes = reinterpret_cast<const char*>(lds);

  f16v acc[kTM][kTN];
#pragma unroll
  for (int i = 0; i < kTM; ++i)
#pragma unroll
    for (int j = 0; j < kTN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  CopyOffsets<BM, kNW> co;
  copy_offsets<BM, kNW>(g, m0, n0, wave, lane, co);
  const ConvSource src(g);
  uint32_t conv_a[BM / 8 / kNW][3];
  if constexpr (CONV == kConvBuffer) {
#pragma unroll
    for (int i = 0; i < BM / 8 / kNW; ++i) {
      const int row = (wave * (BM / 8 / kNW) + i) * 8 + (lane >> 3);
      ConvSource::offsets(g, min(m0 + row, g.m - 1), row, lane & 7, conv_a[i]);
    }
  }
  const FragOffsets fo = frag_offsets<BM>(wm, wn, lr, lg);
  auto issue = [&](int kt, int ring_slot) {  // stage kt's copies into ring slot ring_slot
    const uint32_t dst = lds0 + ring_slot * kStageBytes;
    if constexpr (CONV == kConvAny) {
      dma_stage_conv<BM>(g, m0, n0, kt * kBK, wave, lane, dst);
    } else if constexpr (CONV == kConvBuffer) {
      const int tap = kt * kBK / g.c_in;
#pragma unroll
      for (int i = 0; i < BM / 8 / kNW; ++i)
        src.copy(conv_a[i], tap, kt * kBK, dst + (wave * (BM / 8 / kNW) + i) * 1024);
      dma_stage_w<BM, kNW>(g, co, kt, wave, dst);
    } else {
      dma_stage_s<BM, kNW>(g, co, kt, wave, dst);
    }
  };
  const int kt_n = g.k / kBK;
#pragma unroll
  for (int s = 0; s < kDmaStages; ++s)
    if (s < kt_n) issue(s, s);
  auto main_loop = [&](auto transposed) {
    constexpr bool kT = decltype(transposed)::value;
    Frags<kTM, kTN> fa, fb;
    // this thread's copies of stage kt have landed once at most the later issued stages remain
    wait_stages_ahead<kPerStage, kDmaStages - 1>(min(kDmaStages - 1, kt_n - 1));
    barrier_only();
    load_frags<kTM, kTN>(lds_bytes, fo, fa);
    int cur = 0;  // ring slot of stage kt
    // stage kt with a stage kt + 1 after it
    auto step = [&](int kt, const Frags<kTM, kTN>& frags_kt, Frags<kTM, kTN>& nxt) {
      wait_stages_ahead<kPerStage, kDmaStages - 1>(min(kDmaStages - 2, kt_n - 2 - kt));
      lds_barrier();  // own fragment reads of stage kt done; stage kt + 1 visible; slot kt free
      if (kt + kDmaStages < kt_n) issue(kt + kDmaStages, cur);
      cur = cur + 1 == kDmaStages ? 0 : cur + 1;
      load_frags<kTM, kTN>(lds_bytes + cur * kStageBytes, fo, nxt);
      mma_frags<kTM, kTN, kT>(frags_kt, acc);
    };
    int kt = 0;
    for (; kt + 2 < kt_n; kt += 2) {
      step(kt, fa, fb);
      step(kt + 1, fb, fa);
    }
    if (kt + 1 < kt_n) {
      step(kt, fa, fb);
      mma_frags<kTM, kTN, kT>(fb, acc);
    } else {
      mma_frags<kTM, kTN, kT>(fa, acc);
    }
  };
  if constexpr (EPI == kEpiQkvVt) {
    if (n0 >= 2 * g.q_cols) {  // a v column tile (q_cols % 128 == 0): the branch is uniform per block
      main_loop(std::false_type{});
      store_vt<BM, kTM, kTN, kDmaStages>(g, acc, m0, n0, wm, wn, lr, lg, lds);
      return;
    }
  }
  main_loop(std::true_type{});
  __syncthreads();  // every wave has read its last operand fragments from the ring

  // The tile goes through LDS, so that its rows are written (and the residual's read) 256 bytes at a time:
  // the accumulators give a lane 4 adjacent columns of a row at best, whose stores spread over 32 rows.
  // Against storing from the registers (2 bytes of a column each, 8 bytes on 64-row tiles): a product with
  // a single k stage 4.3 -> 3.8 us at 1500 x 1280, 6.1 -> 5.8 us at 1500 x 3840, 7.45 us as before at
  // 1500 x 5120, where writing 15 MB takes that long either way; the encoder 4034 -> 4012 us.
  // Where it costs: GELU products of short k over many rows (3000 x 5120, k = 320: 28.9 -> 30.1 us).
  if constexpr (EPI == kEpiPartial) {
    constexpr int kRowF = kBN + 4;
    static_assert(BM * kRowF * 4 <= kDmaStages * kStageBytes, "staging tile must fit the ring");
    float* t = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < kTM; ++i)
#pragma unroll
      for (int j = 0; j < kTN; ++j)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          f4v v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * rq + e];
          *reinterpret_cast<f4v*>(t + (wm + 32 * i + lr) * kRowF + wn + 32 * j + 8 * rq + 4 * lg) = v;
        }
    __syncthreads();
#pragma unroll
    for (int c = tid; c < BM * (kBN / 4); c += kNW * 64) {
      const int row = c / (kBN / 4), col = c % (kBN / 4) * 4;
      if (m0 + row < g.m)
        *reinterpret_cast<f4v*>(g.part + (static_cast<size_t>(split) * g.m + m0 + row) * g.n + n0 + col) =
            *reinterpret_cast<const f4v*>(t + row * kRowF + col);
    }
  } else {
    constexpr int kRowH = kBN + 8;  // 16-byte aligned rows
    static_assert(BM * kRowH * 2 <= kDmaStages * kStageBytes, "staging tile must fit the ring");
    _Float16* t = reinterpret_cast<_Float16*>(lds);
#pragma unroll
    for (int j = 0; j < kTN; ++j)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const int cl = wn + 32 * j + 8 * rq + 4 * lg;  // columns cl .. cl + 3 of the tile
        h4u bb = {};
        if (g.bias) bb = *reinterpret_cast<const h4u*>(g.bias + n0 + cl);
#pragma unroll
        for (int i = 0; i < kTM; ++i) {
          h4v o;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = f2h(epilogue_pre<EPI>(acc[i][j][4 * rq + e], h2f(bb[e]), n0 + cl + e, g.q_cols));
          *reinterpret_cast<h4v*>(t + (wm + 32 * i + lr) * kRowH + cl) = o;
        }
      }
    __syncthreads();
#pragma unroll
    for (int c = tid; c < BM * (kBN / 8); c += kNW * 64) {
      const int rl = c / (kBN / 8), cl = c % (kBN / 8) * 8, row = m0 + rl, col = n0 + cl;
      if (row >= g.m) continue;
      h8v v = *reinterpret_cast<const h8v*>(t + rl * kRowH + cl);
      if constexpr (epi_reads_res(EPI)) {
        const h8u r = *reinterpret_cast<const h8u*>(g.res + static_cast<size_t>(row) * g.ldr + col);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = f2h(epilogue_res<EPI>(h2f(v[e]), h2f(r[e])));
      }
      _Float16* dst = EPI == kEpiCrossKV ? g.out + (static_cast<size_t>(col >> 6) * g.t_len + row) * 64 + (col & 63)
                                         : g.out + static_cast<size_t>(row) * g.ldo + col;
      *reinterpret_cast<h8u*>(dst) = v;
    }
  }
}

// ---- 256 x 256 tiles ------------------------------------------------------------------------------
// The cross K/V of 3 or 4 decoder layers: products so wide that 256 x 128 tiles take two passes over the
// CUs. 2 x 4 waves of 128 x 64, a ring of two 64 KB stages; a stage's operands are read 16 of k at a time,
// double-buffered in registers, and the last 16 are multiplied behind the barrier of the next stage, while
// its first are read. A tile moves 2/3 of the bytes per product of a 256 x 128 one and makes 3/4 of
// the LDS reads: MFMAs busy 37% against 31.5%. 1500 x 10240 x 1280: 47.8 -> 41.1 us a call.
constexpr int kWideWaves = 8, kWide = 256, kWideStage = 2 * kWide * 128;
constexpr int kWideRowH = kWide + 8;  // halves per staged output row
constexpr int kWideLds = kWide * kWideRowH * 2 > 2 * kWideStage ? kWide * kWideRowH * 2 : 2 * kWideStage;

__global__ void __launch_bounds__(kWideWaves * 64) gemm_wide_kv_kernel(FW_GEMM_PARAMS) {
  FW_GEMM_TAKE_PARAMS();
  constexpr int kTM = 4, kTN = 2, kCopies = kWide / 8 / kWideWaves;  // copies per wave of each operand
  __shared__ __align__(1024) u32x4 lds[kWideLds / 16];
  int m0, n0;
  tile_origin<kWide, kWide>(g, m0, n0);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave >> 2) * 128, wn = (wave & 3) * 64, lr = lane & 31, lg = lane >> 5;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  uint32_t aoff[kCopies], woff[kCopies];
#pragma unroll
  for (int i = 0; i < kCopies; ++i) {
    const int row = (wave * kCopies + i) * 8 + (lane >> 3), chunk = swz_slot(row, lane & 7) * 8;
    aoff[i] = static_cast<uint32_t>((static_cast<size_t>(min(m0 + row, g.m - 1)) * g.lda + chunk) * 2);
    woff[i] = static_cast<uint32_t>((static_cast<size_t>(n0 + row) * g.ldw + chunk) * 2);
  }
  auto issue = [&](int kt) {
    const uint32_t dst = lds0 + (kt & 1) * kWideStage + wave * kCopies * 1024;
    const size_t kb = static_cast<size_t>(kt) * (kBK * 2);
#pragma unroll
    for (int i = 0; i < kCopies; ++i) dma16_s(aoff[i], reinterpret_cast<const char*>(g.a) + kb, dst + i * 1024);
#pragma unroll
    for (int i = 0; i < kCopies; ++i)
      dma16_s(woff[i], reinterpret_cast<const char*>(g.w) + kb, dst + kWide * 128 + i * 1024);
  };
  const FragOffsets fo = frag_offsets<kWide>(wm, wn, lr, lg);
  struct Step {
    h8v a[kTM], b[kTN];
  };
  auto read = [&](int kt, int s, Step& f) {
    const char* stage = reinterpret_cast<const char*>(lds) + (kt & 1) * kWideStage;
#pragma unroll
    for (int i = 0; i < kTM; ++i) f.a[i] = *reinterpret_cast<const h8v*>(stage + fo.a[s] + 4096 * i);
#pragma unroll
    for (int j = 0; j < kTN; ++j) f.b[j] = *reinterpret_cast<const h8v*>(stage + fo.b[s] + 4096 * j);
  };
  f16v acc[kTM][kTN];
#pragma unroll
  for (int i = 0; i < kTM; ++i)
#pragma unroll
    for (int j = 0; j < kTN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  auto multiply = [&](const Step& f) {
#pragma unroll
    for (int i = 0; i < kTM; ++i)
#pragma unroll
      for (int j = 0; j < kTN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.b[j], f.a[i], acc[i][j], 0, 0, 0);
  };
  const int kt_n = g.k / kBK;
  // stage kt has landed and every wave sees it; every wave has read stage kt - 1, whose slot is refilled
  auto enter = [&](int kt) {
    wait_vmcnt<0>();
    lds_barrier();
    if (kt + 1 < kt_n) issue(kt + 1);
  };
  Step f0, f1;
  issue(0);
  enter(0);
  read(0, 0, f0);
  for (int kt = 0; kt < kt_n; ++kt) {
    read(kt, 1, f1);
    multiply(f0);
    read(kt, 2, f0);
    multiply(f1);
    read(kt, 3, f1);
    multiply(f0);
    if (kt + 1 < kt_n) {
      enter(kt + 1);
      read(kt + 1, 0, f0);
    }
    multiply(f1);
  }
  __syncthreads();  // every wave has read its last operands
  _Float16* t = reinterpret_cast<_Float16*>(lds);
#pragma unroll
  for (int j = 0; j < kTN; ++j)
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      const int cl = wn + 32 * j + 8 * rq + 4 * lg;  // columns cl .. cl + 3 of the tile
      h4u bb = {};
      if (g.bias) bb = *reinterpret_cast<const h4u*>(g.bias + n0 + cl);
#pragma unroll
      for (int i = 0; i < kTM; ++i) {
        h4v o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = f2h(acc[i][j][4 * rq + e] + h2f(bb[e]));
        *reinterpret_cast<h4v*>(t + (wm + 32 * i + lr) * kWideRowH + cl) = o;
      }
    }
  __syncthreads();
#pragma unroll 4
  for (int c = tid; c < kWide * (kWide / 8); c += kWideWaves * 64) {
    const int rl = c / (kWide / 8), cl = c % (kWide / 8) * 8, row = m0 + rl, col = n0 + cl;
    if (row < g.m)
      *reinterpret_cast<h8u*>(g.out + (static_cast<size_t>(col >> 6) * g.t_len + row) * 64 + (col & 63)) =
          *reinterpret_cast<const h8v*>(t + rl * kWideRowH + cl);
  }
}

// ---- k-sliced GEMM for few rows ----------------------------------------------------------------
// out = epilogue(A W^T) where the tiles of gemm_dma_kernel would leave most CUs idle. A block's kKsWaves
// waves all compute the whole TM x TN tile, wave w over the 64-wide k stages w, w + kKsWaves, ...: each
// wave fills and reads a ring of its own, so the main loop has no barrier, and a stage's operands are
// read from LDS once (waves that split the tile read the A or W half they share again: 64-row tiles of
// 32 x 32 waves spend 512 LDS clocks a stage on 128 clocks of MFMA). The waves' sums are added in wave
// order through LDS, then the epilogue runs on 4 adjacent columns a thread. What bounds it is the weights'
// way from HBM: 128 KB or more in flight per CU. A 4-layer encoder over 251 frames, stem and cross K/V:
// 424 -> 309 us (fc2 20.2 -> 12.3, out 10.7 -> 6.7 us a launch).
constexpr int kKsWaves = 4;
constexpr int kKsLds = 160 * 1024;
template <int TM, int TN>
constexpr int ks_stages() {  // ring depth per wave: what fits one block's LDS, at most 4
  return kKsLds / (kKsWaves * (TM + TN) * 128) < 4 ? kKsLds / (kKsWaves * (TM + TN) * 128) : 4;
}

template <int TM, int TN, int EPI, bool CONV>
__global__ void __launch_bounds__(kKsWaves * 64) gemm_ks_kernel(FW_GEMM_PARAMS) {
  FW_GEMM_TAKE_PARAMS();
  constexpr int kST = ks_stages<TM, TN>(), kTM = TM / 32, kTN = TN / 32;
  constexpr int kStageBytes = (TM + TN) * 128, kPer = (TM + TN) / 8;  // copies per stage
  constexpr int kRowF = TN + 4;                                      // floats per staged row of sums
  static_assert(kST >= 2 && (kST - 1) * kPer < 64, "ring depth");
  static_assert(TM * kRowF * 4 <= kST * kStageBytes, "a wave's sums fit its ring");
  __shared__ __align__(1024) u32x4 lds[kKsWaves * kST * kStageBytes / 16];

  int m0, n0;
  tile_origin<TM, TN>(g, m0, n0);
  int split = 0;
  if constexpr (EPI == kEpiPartial) {
    split = static_cast<int>(blockIdx.x) / ((g.n / TN) * ((g.m + TM - 1) / TM));
    g.a += static_cast<size_t>(split) * g.k;
    g.w += static_cast<size_t>(split) * g.k;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lg = lane >> 5, rsub = lane >> 3, slot8 = lane & 7;
  char* ring = reinterpret_cast<char*>(lds) + wave * (kST * kStageBytes);
  const uint32_t ring0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(ring));

  // byte offsets of this lane's chunk of every copy of a stage (A rows, then W rows)
  uint32_t aoff[TM / 8][3], woff[TN / 8];
  const ConvSource src(g);
#pragma unroll
  for (int i = 0; i < TM / 8; ++i) {
    const int row = i * 8 + rsub, gm = min(m0 + row, g.m - 1);
    if constexpr (CONV)
      ConvSource::offsets(g, gm, row, slot8, aoff[i]);
    else
      aoff[i][0] = static_cast<uint32_t>((static_cast<size_t>(gm) * g.lda + swz_slot(row, slot8) * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < TN / 8; ++i) {
    const int row = i * 8 + rsub;
    woff[i] = static_cast<uint32_t>((static_cast<size_t>(n0 + row) * g.ldw + swz_slot(row, slot8) * 8) * 2);
  }
  auto issue = [&](int kt, int slot) {
    const uint32_t dst = __builtin_amdgcn_readfirstlane(ring0 + slot * kStageBytes);
    const size_t kb = static_cast<size_t>(kt) * (kBK * 2);
    if constexpr (CONV) {
      const int tap = kt * kBK / g.c_in;
#pragma unroll
      for (int i = 0; i < TM / 8; ++i) src.copy(aoff[i], tap, kt * kBK, dst + i * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < TM / 8; ++i) dma16_s(aoff[i][0], reinterpret_cast<const char*>(g.a) + kb, dst + i * 1024);
    }
#pragma unroll
    for (int i = 0; i < TN / 8; ++i)
      dma16_s(woff[i], reinterpret_cast<const char*>(g.w) + kb, dst + TM * 128 + i * 1024);
  };
  const FragOffsets fo = frag_offsets<TM>(0, 0, lr, lg);
  f16v acc[kTM][kTN];
#pragma unroll
  for (int i = 0; i < kTM; ++i)
#pragma unroll
    for (int j = 0; j < kTN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int kt_all = g.k / kBK, n_st = (kt_all - wave + kKsWaves - 1) / kKsWaves;  // this wave's stages
#pragma unroll
  for (int s = 0; s < kST; ++s)
    if (s < n_st) issue(wave + s * kKsWaves, s);
  if (n_st > 0) {
    Frags<kTM, kTN> fa, fb;
    wait_stages_ahead<kPer, kST - 1>(min(kST - 1, n_st - 1));
    load_frags<kTM, kTN>(ring, fo, fa);
    int cur = 0;
    auto step = [&](int i, const Frags<kTM, kTN>& now, Frags<kTM, kTN>& nxt) {
      wait_stages_ahead<kPer, kST - 1>(min(kST - 2, n_st - 2 - i));
      lds_reads_done();  // stage i is in registers: its slot is free
      if (i + kST < n_st) issue(wave + (i + kST) * kKsWaves, cur);
      cur = cur + 1 == kST ? 0 : cur + 1;
      load_frags<kTM, kTN>(ring + cur * kStageBytes, fo, nxt);
      mma_frags<kTM, kTN, true>(now, acc);
    };
    int i = 0;
    for (; i + 2 < n_st; i += 2) {
      step(i, fa, fb);
      step(i + 1, fb, fa);
    }
    if (i + 1 < n_st) {
      step(i, fa, fb);
      mma_frags<kTM, kTN, true>(fb, acc);
    } else {
      mma_frags<kTM, kTN, true>(fa, acc);
    }
  }
  // this wave's sums, row by row, into its own ring (every copy has landed and been read)
  lds_reads_done();
  float* sums = reinterpret_cast<float*>(ring);
#pragma unroll
  for (int i = 0; i < kTM; ++i)
#pragma unroll
    for (int j = 0; j < kTN; ++j)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        f4v v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * rq + e];
        *reinterpret_cast<f4v*>(sums + (32 * i + lr) * kRowF + 32 * j + 8 * rq + 4 * lg) = v;
      }
  __syncthreads();
  const float* part0 = reinterpret_cast<const float*>(lds);
  constexpr int kWaveF = kST * kStageBytes / 4;  // floats between the waves' sums
  if constexpr (EPI == kEpiQkvVt) {
    if (n0 >= 2 * g.q_cols) {  // a tile of v columns: 4 adjacent keys of one column per thread, stored transposed
      _Float16* dst = g.vt + static_cast<size_t>(n0 - 2 * g.q_cols) * g.vt_pad;
      // a wave takes 16 keys of 16 columns at a time: its reads of the sums meet in no LDS bank (4 rows are 16
      // banks on), and 4 lanes store 32 bytes of a column (a column's 64 keys a quarter-wave: every read 4-way)
      static_assert(4 * kRowF % 64 == 16, "4 rows of sums are 16 banks on");
#pragma unroll
      for (int c = tid; c < TM / 4 * TN; c += kKsWaves * 64) {
        const int blk = c >> 6, col = blk / (TM / 16) * 16 + (c >> 2 & 15);
        const int rl = blk % (TM / 16) * 16 + (c & 3) * 4;  // rows rl .. rl + 3 stay adjacent under vt_pos
        const float b = g.bias ? h2f(g.bias[n0 + col]) : 0.f;
        h4v o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float v = 0.f;
#pragma unroll
          for (int w = 0; w < kKsWaves; ++w) v += part0[w * kWaveF + (rl + e) * kRowF + col];
          o[e] = m0 + rl + e < g.m ? f2h(v + b) : static_cast<_Float16>(0.f);
        }
        if (m0 + rl < g.vt_pad) *reinterpret_cast<h4v*>(dst + static_cast<size_t>(col) * g.vt_pad + m0 + vt_pos(rl)) = o;
      }
      // the last row tile may end before V^T's padding to whole 64-key tiles: zeros from there on
      const int pad4 = m0 + TM >= g.m ? (g.vt_pad - m0 - TM) / 4 : 0;
      for (int c = tid; c < pad4 * TN; c += kKsWaves * 64)
        *reinterpret_cast<h4v*>(dst + static_cast<size_t>(c / pad4) * g.vt_pad + m0 + TM + c % pad4 * 4) = h4v{};
      return;
    }
  }
  constexpr int kCols4 = TN / 4;
#pragma unroll
  for (int c = tid; c < TM * kCols4; c += kKsWaves * 64) {
    const int rl = c / kCols4, cl = c % kCols4 * 4, row = m0 + rl, col = n0 + cl;
    f4v v = *reinterpret_cast<const f4v*>(part0 + rl * kRowF + cl);
#pragma unroll
    for (int w = 1; w < kKsWaves; ++w) {
      const f4v u = *reinterpret_cast<const f4v*>(part0 + w * kWaveF + rl * kRowF + cl);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += u[e];
    }
    if (row >= g.m) continue;
    if constexpr (EPI == kEpiPartial) {
      *reinterpret_cast<f4v*>(g.part + (static_cast<size_t>(split) * g.m + row) * g.n + col) = v;
    } else {
      h4u bb = {};
      h4v o;
      if (g.bias) bb = *reinterpret_cast<const h4u*>(g.bias + col);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = epilogue_pre<EPI>(v[e], h2f(bb[e]), col + e, g.q_cols);
      if constexpr (epi_reads_res(EPI)) {
        const h4u rv = *reinterpret_cast<const h4u*>(g.res + static_cast<size_t>(row) * g.ldr + col);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = epilogue_res<EPI>(v[e], h2f(rv[e]));
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = f2h(v[e]);
      if constexpr (EPI == kEpiCrossKV)
        *reinterpret_cast<h4u*>(g.out + (static_cast<size_t>(col >> 6) * g.t_len + row) * 64 + (col & 63)) = o;
      else
        *reinterpret_cast<h4u*>(g.out + static_cast<size_t>(row) * g.ldo + col) = o;
    }
  }
}

#ifndef FW_XCD_GROUP
#define FW_XCD_GROUP 1
#endif
static_assert(FW_XCD_GROUP == 0 || FW_XCD_GROUP == 1, "FW_XCD_GROUP is a switch (0 or 1)");
// Picks the XCD rectangle grid that divides the tile grid and moves the fewest bytes into the L2s:
// A is fetched once per column group (xn), W once per row group (xm). Convs too where their weights exceed
// an L2 (3000 -> 1500 x 1280, k = 3840: 27.2 -> 26.6 us, 1280 -> 640: 21.4 -> 19.3 us); with the short k of
// the first conv the row-major order is faster (1280 rows: 6.8 against 7.0 us).
void choose_xcd_groups(GemmArgs& g, int bm, int bn = kBN) {
  g.xm = g.xn = 0;
  if (!FW_XCD_GROUP || (g.conv_stride && g.k < 1024)) return;
  const int ntm = (g.m + bm - 1) / bm, ntn = g.n / bn;
  double best = 0;
  for (int xm = 1; xm <= 8; xm *= 2) {
    const int xn = 8 / xm;
    if (ntm % xm || ntn % xn) continue;
    const double bytes = static_cast<double>(xn) * g.m * g.k + static_cast<double>(xm) * g.n * g.k;
    if (!g.xm || bytes < best) {
      best = bytes;
      g.xm = xm;
      g.xn = xn;
    }
  }
}

// The plain GEMMs address each operand as a scalar base plus a 32-bit per-lane byte offset
// (dma_stage_s): the rows a block reads must lie within 4 GiB of the operand's start.
bool copy_offsets_fit(const GemmArgs& g) {
  constexpr size_t kLimit = static_cast<size_t>(1) << 32;
  return (static_cast<size_t>(g.m - 1) * g.lda + kBK) * 2 < kLimit &&
         (static_cast<size_t>(g.n - 1) * g.ldw + kBK) * 2 < kLimit;
}

template <int BM, int CONV, int ST = dma_stages<BM>()>
int launch_dma(GemmArgs g, int epi, hipStream_t s) {
  const dim3 grid((g.n / kBN) * ((g.m + BM - 1) / BM)), block(gemm_waves<BM>() * 64);
  choose_xcd_groups(g, BM);
  switch (epi) {
#define FW_GEMM_CASE(E, C) \
  case E:                  \
    if constexpr (C || CONV == kNoConv) hipLaunchKernelGGL((gemm_dma_kernel<BM, E, CONV, ST>), grid, block, 0, s, FW_GEMM_ARGS(g)); \
    break;
    FW_GEMM_CASE(FW_EPI_BIAS, true)
    FW_GEMM_CASE(FW_EPI_BIAS_GELU, true)
    FW_GEMM_CASE(FW_EPI_BIAS_GELU_POS, true)
    FW_GEMM_CASE(FW_EPI_BIAS_RESID, false)
    FW_GEMM_CASE(FW_EPI_BIAS_RESID_CLAMP, false)
    FW_GEMM_CASE(FW_EPI_SCALE_Q, false)
    FW_GEMM_CASE(kEpiCrossKV, false)
    FW_GEMM_CASE(kEpiQkvVt, false)
#undef FW_GEMM_CASE
    default:
      return fw_fail(FW_EINVAL, "gemm: unknown epilogue %d", epi);
  }
  return fw_check_launch(CONV ? "conv1d" : "gemm");
}

template <int TM, int TN, bool CONV>
int launch_ks(GemmArgs g, int epi, hipStream_t s) {
  const dim3 grid((g.n / TN) * ((g.m + TM - 1) / TM)), block(kKsWaves * 64);
  choose_xcd_groups(g, TM, TN);
  switch (epi) {
#define FW_KS_CASE(E, C) \
  case E:                \
    if constexpr (C) hipLaunchKernelGGL((gemm_ks_kernel<TM, TN, E, CONV>), grid, block, 0, s, FW_GEMM_ARGS(g)); \
    break;
    FW_KS_CASE(FW_EPI_BIAS, true)
    FW_KS_CASE(FW_EPI_BIAS_GELU, true)
    FW_KS_CASE(FW_EPI_BIAS_GELU_POS, true)
    FW_KS_CASE(FW_EPI_BIAS_RESID, !CONV)
    FW_KS_CASE(FW_EPI_BIAS_RESID_CLAMP, !CONV)
    FW_KS_CASE(FW_EPI_SCALE_Q, !CONV)
    FW_KS_CASE(kEpiCrossKV, !CONV)
    FW_KS_CASE(kEpiQkvVt, !CONV)
#undef FW_KS_CASE
    default:
      return fw_fail(FW_EINVAL, "gemm: unknown epilogue %d", epi);
  }
  return fw_check_launch(CONV ? "conv1d" : "gemm");
}

template <int TM, int TN>
int launch_ks_partial(GemmArgs g, hipStream_t s) {
  const dim3 grid((g.n / TN) * ((g.m + TM - 1) / TM) * g.splits);
  choose_xcd_groups(g, TM, TN);
  hipLaunchKernelGGL((gemm_ks_kernel<TM, TN, kEpiPartial, false>), grid, dim3(kKsWaves * 64), 0, s, FW_GEMM_ARGS(g));
  return fw_check_launch("gemm_splitk");
}

// The tile: the fewest passes over the CUs (one block per CU: each tile's ring takes most of its LDS) at
// the tile's cost, kPassUs + k stages x per_stage. Both are fits to times on MI355X with weights cold (a
// graph over >300 MB of them; m = 50 .. 1500, n = 1280, 3840, 5120, k = 1280, 2 x 2560 and the convs'
// 3840). The absolute times are rough: over 15 row counts of 7 products the picked tile took 0.67 to 1.25 times
// what the fit says, the low end where launches are shortest. What decides is mostly the passes: the pick was
// the fastest or within 2% of it, but for fc2 at 577 and 640 rows (64x64 6% and 9% faster than its 128x128).
// 96 x 64 serves the split products: of a whole one's 64 x 128 tiles there are never more, and they cost no more.
// Measured us for (m, n, k) by tile:
//   (50, 1280, 1280)   32x32 4.8, 64x32 6.2, 64x64 7.8, 64x128 9.6
//   (251, 1280, 1280)  32x32 7.8 (2 passes), 64x32 6.3, 64x64 8.2, 64x128 10.5, 128x128 15.1
//   (251, 5120, 1280)  64x64 19.6 (2), 96x64 14.0, 64x128 14.4, 128x128 18.7 (weights in L2: 96x64 11.3, 64x128 9.9)
//   (1000, 1280, 1280) 96x64 12.8, 64x128 10.7
//   (640, 5120, 1280)  64x128 26 (2), 128x128 19.0, 192x128 21.9, 256x128 26.2
//   (1000, 3840, 1280) 64x128 24.2 (2), 128x128 18.1, 192x128 19.6, 256x128 24.6
//   (1200, 5120, 1280) 128x128 34.3 (2), 192x128 38.0 (2), 256x128 30.4
//   (251, 1280, 2 x 2560) 64x32 19.4 (2), 64x64 15.1, 96x64 17.7, 128x128 28.4
//   (400, 1280, 2 x 2560) 64x64 26.1 (2), 96x64 17.6, 128x128 23.1
// A conv's stage costs what a plain product's does: its sources are per-lane offsets too. The stem's second
// conv, (769 / 900 / 1000 / 1152, 1280, 3840): 96x64 29.4 / 28.5 / 29.5 / 29.1, 64x128 26.8 / 27.1 / 29.8 / 31.2.
enum Tile { kD256, kD192, kD128, kD64, kS96x64, kS64x64, kS64x32, kS32x32, kWide256, kTiles };
struct TileCost {
  int rows, cols;
  float per_stage;  // us per 64-wide k stage and pass
};
constexpr TileCost kTileCost[kTiles] = {{256, 128, 1.15f}, {192, 128, 0.85f}, {128, 128, 0.62f}, {64, 128, 0.42f},
                                        {96, 64, 0.43f},   {64, 64, 0.28f},   {64, 32, 0.18f},   {32, 32, 0.11f},
                                        {kWide, kWide, 1.55f}};
constexpr float kPassUs = 4.f;
constexpr int kCus = 256;

// What the fit leaves out, us by both tiles:
//  - 64 x 64 and 96 x 64 sliced tiles with fewer k stages than waves: the idle waves' sums are added all the same
//    ((400, 1280, 64) 64x64 4.9, 64x128 4.5; (6000, 128, 2 x 64) 96x64 5.3, 128x128 4.5; four stages even).
//  - q/k/v on 64 x 64 sliced tiles: kVtUs a pass for V^T, stored 8 bytes a lane ((500, 1152, 384) 5.6, 64x128 5.2;
//    (333, 1536, 512) 6.1, 6.1; (251, 3840, 1280) 10.6, 13.4). Its unfused form too, so that both give the same bits.
//  - Three passes or more of 256-row tiles cost less than that many single ones: they stay up to kManyPasses of
//    the best ((8000, 3840, 1280) 113, 192x128 120; (8000, 2560, 5120) 239, 192x128 254, 128x128 256).
constexpr float kVtUs = 1.5f, kManyPasses = 1.08f;

template <class Allowed>
Tile choose_tile(const GemmArgs& g, Allowed allowed, bool vt = false) {
  Tile best = kD128;
  float best_us = 0.f;
  const bool few_stages = g.k < kKsWaves * kBK;
  for (int t = kTiles - 1; t >= 0; --t) {  // the 256-row tile last
    if (!allowed(static_cast<Tile>(t)) || (few_stages && (t == kS64x64 || t == kS96x64))) continue;
    const TileCost& c = kTileCost[t];
    const int64_t blocks = static_cast<int64_t>(g.n / c.cols) * ((g.m + c.rows - 1) / c.rows) * (g.splits > 1 ? g.splits : 1);
    const int64_t passes = (blocks + kCus - 1) / kCus;
    const float pass_us = kPassUs + static_cast<float>(g.k / kBK) * c.per_stage + (vt && t == kS64x64 ? kVtUs : 0.f);
    const float us = static_cast<float>(passes) * pass_us;
    if (best_us == 0.f || us <= best_us || (t == kD256 && passes >= 3 && us < kManyPasses * best_us)) {
      best = static_cast<Tile>(t);
      best_us = us;
    }
  }
  return best;
}

int launch_gemm(const GemmArgs& g, int epi, hipStream_t s) {
  if (!copy_offsets_fit(g)) return fw_fail(FW_EINVAL, "gemm: each operand must span less than 4 GiB");
  const bool wide = epi == kEpiCrossKV && g.n % kWide == 0;  // the one epilogue that the wide tiles have
  switch (choose_tile(g, [&](Tile t) { return t != kS96x64 && (t != kWide256 || wide); },
                      epi == kEpiQkvVt || epi == FW_EPI_SCALE_Q)) {
    case kD256: return launch_dma<256, kNoConv>(g, epi, s);
    case kD192: return launch_dma<192, kNoConv>(g, epi, s);
    case kD64: return launch_dma<64, kNoConv>(g, epi, s);
    case kS64x64: return launch_ks<64, 64, false>(g, epi, s);
    case kS64x32: return launch_ks<64, 32, false>(g, epi, s);
    case kS32x32: return launch_ks<32, 32, false>(g, epi, s);
    case kWide256: {
      GemmArgs w = g;
      choose_xcd_groups(w, kWide, kWide);
      hipLaunchKernelGGL(gemm_wide_kv_kernel, dim3((g.n / kWide) * ((g.m + kWide - 1) / kWide)), dim3(kWideWaves * 64), 0, s,
                         FW_GEMM_ARGS(w));
      return fw_check_launch("gemm");
    }
    default: return launch_dma<128, kNoConv>(g, epi, s);
  }
}

// Convs. With a short k (the 128 -> 1280 conv of the stem, k = 384: six stages) a pass is mostly fill,
// drain and epilogue: past one pass of 64 x 64 tiles, 64-row tiles with a 3-deep ring, two blocks on a
// CU, so that one's epilogue runs beside the other's copies (3000 rows: 9.9 us against 12.6 for a
// register-staged gather, 10.3 for a 2-deep ring and 10.1 for 128-row tiles; 1000 rows: 6.7, 10.5, 7.8, 9.4).
int launch_conv(const GemmArgs& g, int epi, hipStream_t s) {
  if (!conv_offsets_fit(g) || !copy_offsets_fit(g)) return launch_dma<128, kConvAny>(g, epi, s);
  switch (choose_tile(g, [&](Tile t) { return t >= kD128 && t != kS96x64 && t != kWide256; })) {
    case kS64x64: return launch_ks<64, 64, true>(g, epi, s);
    case kS64x32: return launch_ks<64, 32, true>(g, epi, s);
    case kS32x32: return launch_ks<32, 32, true>(g, epi, s);
    case kD64:
      if (g.k >= 1024) return launch_dma<64, kConvBuffer>(g, epi, s);
      break;
    default:
      if (g.k >= 1024) return launch_dma<128, kConvBuffer>(g, epi, s);
  }
  return launch_dma<64, kConvBuffer, 3>(g, epi, s);
}

// ------------------------------------------------------------------------------------------
// Row LayerNorm over 1280 columns: 32 lanes per row (5 x 16-byte chunks each), kLnRows = kLnThreads / 32 rows per block.
// ------------------------------------------------------------------------------------------
constexpr int kLnC = kHidden / 8 / 32;  // 16-byte fp16 chunks per lane of a row
// One wave (two rows) a block for both kernels: 251 rows make 126 blocks instead of 32. Four encoder layers over
// 251 frames take 245.3 us, with 256 threads in both 249.9, in the plain one alone 246.9, in the residual one
// alone 249.1; over 50 frames 157.5 and 161.0; over 500 to 1500 frames all within 0.5%. Chains of either alone
// are the fastest at 64 threads from 1 to 20000 rows (1500 rows: plain 3.5 against 3.7 us, residual 5.1, 5.6).
#ifndef FW_LN_THREADS
#define FW_LN_THREADS 64
#endif
constexpr int kLnThreads = FW_LN_THREADS;  // threads per row-LayerNorm block: 32 lanes per row
constexpr int kLnRows = kLnThreads / 32;
static_assert(kLnThreads % 64 == 0 && kLnThreads <= 256, "whole waves, within the launch bounds");

// LayerNorm of one row held as v[] (this lane's elements: chunks sub + 32 c) with gamma / beta chunks
// gu / bu, written to yr when valid.
__device__ __forceinline__ void ln_row_finish(const float (&v)[kLnC * 8], const uint4 (&gu)[kLnC],
                                              const uint4 (&bu)[kLnC], float eps, uint4* yr, bool valid, int sub) {
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kLnC * 8; ++i) sum += v[i];
  const float mean = group_sum<32>(sum) * (1.0f / kHidden);
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < kLnC * 8; ++i) {
    const float d = v[i] - mean;
    sq += d * d;
  }
  const float inv = rsqrtf(group_sum<32>(sq) * (1.0f / kHidden) + eps);
#pragma unroll
  for (int c = 0; c < kLnC; ++c) {
    const _Float16* gp = reinterpret_cast<const _Float16*>(&gu[c]);
    const _Float16* bp = reinterpret_cast<const _Float16*>(&bu[c]);
    uint4 o;
    _Float16* op = reinterpret_cast<_Float16*>(&o);
#pragma unroll
    for (int e = 0; e < 8; ++e) op[e] = f2h((v[c * 8 + e] - mean) * inv * h2f(gp[e]) + h2f(bp[e]));
    // computed outside the store's lane mask, so the gamma / beta requests are not sunk into it
    asm volatile("" : "+v"(o.x), "+v"(o.y), "+v"(o.z), "+v"(o.w));
    if (valid) yr[sub + 32 * c] = o;
  }
}

__global__ void __launch_bounds__(256) layernorm_rows_kernel(const _Float16* __restrict__ x,
                                                             const _Float16* __restrict__ gamma,
                                                             const _Float16* __restrict__ beta,
                                                             _Float16* __restrict__ y, int rows, float eps) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sub = lane & 31;
  const int row = blockIdx.x * kLnRows + wave * 2 + (lane >> 5);
  const bool valid = row < rows;
  const uint4* xr = reinterpret_cast<const uint4*>(x + static_cast<size_t>(valid ? row : 0) * kHidden);
  // gamma and beta are requested with the row, not after the two reductions
  const uint4* g4 = reinterpret_cast<const uint4*>(gamma);
  const uint4* b4 = reinterpret_cast<const uint4*>(beta);
  uint4 xu[kLnC], gu[kLnC], bu[kLnC];
#pragma unroll
  for (int c = 0; c < kLnC; ++c) xu[c] = xr[sub + 32 * c];
#pragma unroll
  for (int c = 0; c < kLnC; ++c) {
    gu[c] = g4[sub + 32 * c];
    bu[c] = b4[sub + 32 * c];
  }
  float v[kLnC * 8];
#pragma unroll
  for (int c = 0; c < kLnC; ++c) {
    const _Float16* hp = reinterpret_cast<const _Float16*>(&xu[c]);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[c * 8 + e] = h2f(hp[e]);
  }
  ln_row_finish(v, gu, bu, eps, reinterpret_cast<uint4*>(y + static_cast<size_t>(valid ? row : 0) * kHidden), valid,
                sub);
}

// The end of a split-k product followed by a LayerNorm: the split sums part[0 .. 1] of row r are added
// (in split order), then the residual epilogue of fw_gemm (FW_EPI_BIAS_RESID, or with CLAMP
// FW_EPI_BIAS_RESID_CLAMP) updates h[r] in place, and y[r] <- LN(h[r]) exactly as layernorm_rows_kernel.
template <bool CLAMP>
__global__ void __launch_bounds__(256) residual_layernorm_rows_kernel(const float* __restrict__ part,
                                                                      const _Float16* __restrict__ bias,
                                                                      _Float16* h,
                                                                      const _Float16* __restrict__ gamma,
                                                                      const _Float16* __restrict__ beta,
                                                                      _Float16* __restrict__ y, int rows, float eps) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sub = lane & 31;
  const int row = blockIdx.x * kLnRows + wave * 2 + (lane >> 5);
  const bool valid = row < rows;
  const size_t r0 = static_cast<size_t>(valid ? row : 0) * kHidden;
  const size_t split_stride = static_cast<size_t>(rows) * kHidden;
  const float4* p0 = reinterpret_cast<const float4*>(part + r0);
  const float4* p1 = reinterpret_cast<const float4*>(part + split_stride + r0);
  uint4* hr = reinterpret_cast<uint4*>(h + r0);
  const uint4* g4 = reinterpret_cast<const uint4*>(gamma);
  const uint4* b4 = reinterpret_cast<const uint4*>(beta);
  const uint4* bi4 = reinterpret_cast<const uint4*>(bias);
  uint4 hu[kLnC], gu[kLnC], bu[kLnC], biu[kLnC];
  float4 a0[kLnC][2], a1[kLnC][2];
#pragma unroll
  for (int c = 0; c < kLnC; ++c) {
    const int q = sub + 32 * c;  // this lane's 8-element chunk
    a0[c][0] = p0[2 * q];
    a0[c][1] = p0[2 * q + 1];
    a1[c][0] = p1[2 * q];
    a1[c][1] = p1[2 * q + 1];
    hu[c] = hr[q];
  }
#pragma unroll
  for (int c = 0; c < kLnC; ++c) {
    gu[c] = g4[sub + 32 * c];
    bu[c] = b4[sub + 32 * c];
    biu[c] = bi4[sub + 32 * c];
  }
  float v[kLnC * 8];
#pragma unroll
  for (int c = 0; c < kLnC; ++c) {
    const _Float16* rp = reinterpret_cast<const _Float16*>(&hu[c]);
    const _Float16* bp = reinterpret_cast<const _Float16*>(&biu[c]);
    const float* s0 = reinterpret_cast<const float*>(&a0[c][0]);
    const float* s1 = reinterpret_cast<const float*>(&a1[c][0]);
    uint4 o;
    _Float16* op = reinterpret_cast<_Float16*>(&o);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float acc = s0[e] + s1[e];
      float t = round_h(acc + h2f(bp[e]));
      if constexpr (CLAMP) {
        t = round_h(h2f(rp[e]) + t);
        const float lim = 65504.0f - 1000.0f;
        // the LayerNorm below reads the stored fp16 value: the bound itself rounds to 64512
        t = round_h(fminf(fmaxf(t, -lim), lim));
      } else {
        t = round_h(h2f(rp[e]) + t);
      }
      op[e] = f2h(t);
      v[c * 8 + e] = t;
    }
    asm volatile("" : "+v"(o.x), "+v"(o.y), "+v"(o.z), "+v"(o.w));
    if (valid) hr[sub + 32 * c] = o;
  }
  ln_row_finish(v, gu, bu, eps, reinterpret_cast<uint4*>(y + r0), valid, sub);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
bool aligned8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }

}  // namespace
}  // namespace fw

using namespace fw;

extern "C" int fw_gemm(const void* a, int lda, const void* w, int ldw, const void* bias, void* out, int ldo,
                       const void* res, int ldr, int m, int n, int k, int epilogue, int q_cols, hipStream_t stream) {
  if (!a || !w || !out) return fw_fail(FW_EINVAL, "gemm: null pointer");
  if (m <= 0 || n <= 0 || k <= 0 || n % kBN || k % kBK)
    return fw_fail(FW_EINVAL, "gemm: need m > 0, n %% %d == 0, k %% %d == 0 (m=%d n=%d k=%d)", kBN, kBK, m, n, k);
  if (lda < k || ldw < k || ldo < n || lda % 8 || ldw % 8 || ldo % 8 || !aligned16(a) || !aligned16(w))
    return fw_fail(FW_EINVAL, "gemm: leading dimensions must cover the matrix and be multiples of 8");
  const bool needs_res = epilogue == FW_EPI_BIAS_RESID || epilogue == FW_EPI_BIAS_RESID_CLAMP ||
                         epilogue == FW_EPI_BIAS_GELU_POS;
  if (needs_res && (!res || ldr < n)) return fw_fail(FW_EINVAL, "gemm: epilogue %d needs res with ldr >= n", epilogue);
  if (!aligned8(out) || (bias && !aligned8(bias)) || (needs_res && (!aligned8(res) || ldr % 8)))
    return fw_fail(FW_EINVAL, "gemm: out, bias and res must be 8-byte aligned (and ldr a multiple of 8)");
  if (epilogue < FW_EPI_BIAS || epilogue > FW_EPI_SCALE_Q) return fw_fail(FW_EINVAL, "gemm: unknown epilogue %d", epilogue);
  GemmArgs g{static_cast<const _Float16*>(a), lda, static_cast<const _Float16*>(w), ldw,
             static_cast<const _Float16*>(bias), static_cast<_Float16*>(out), ldo,
             static_cast<const _Float16*>(res), ldr, m, n, k, q_cols, 0, 0, 0, 0, 0};
  return launch_gemm(g, epilogue, stream);
}

extern "C" int fw_conv1d(const void* x, int t_in, int c_in, int stride, const void* wp, const void* bias, void* out,
                         int c_out, const void* res, int epilogue, hipStream_t stream) {
  if (!x || !wp || !out) return fw_fail(FW_EINVAL, "conv1d: null pointer");
  if (t_in <= 0 || c_in <= 0 || c_in % 64 || c_out % kBN || (stride != 1 && stride != 2))
    return fw_fail(FW_EINVAL, "conv1d: need c_in %% 64 == 0, c_out %% %d == 0, stride 1 or 2", kBN);
  if (epilogue != FW_EPI_BIAS_GELU && epilogue != FW_EPI_BIAS_GELU_POS && epilogue != FW_EPI_BIAS)
    return fw_fail(FW_EINVAL, "conv1d: unsupported epilogue %d", epilogue);
  if (epilogue == FW_EPI_BIAS_GELU_POS && !res) return fw_fail(FW_EINVAL, "conv1d: positions required");
  if (!aligned16(x) || !aligned16(wp)) return fw_fail(FW_EINVAL, "conv1d: x and wp must be 16-byte aligned");
  const int t_out = (t_in - 1) / stride + 1;
  GemmArgs g{static_cast<const _Float16*>(x), c_in, static_cast<const _Float16*>(wp), 3 * c_in,
             static_cast<const _Float16*>(bias), static_cast<_Float16*>(out), c_out,
             static_cast<const _Float16*>(res), c_out, t_out, c_out, 3 * c_in, 0, stride, t_in, c_in, 0, 0};
  return launch_conv(g, epilogue, stream);
}

extern "C" int fw_layernorm_rows(const void* x, const void* gamma, const void* beta, void* y, int rows, int n,
                                 float eps, hipStream_t stream) {
  if (!x || !gamma || !beta || !y) return fw_fail(FW_EINVAL, "layernorm_rows: null pointer");
  if (n != kHidden || rows <= 0) return fw_fail(FW_EINVAL, "layernorm_rows: n must be %d", kHidden);
  if (!aligned16(x) || !aligned16(y) || !aligned16(gamma) || !aligned16(beta))
    return fw_fail(FW_EINVAL, "layernorm_rows: tensors must be 16-byte aligned");
  hipLaunchKernelGGL(layernorm_rows_kernel, dim3((rows + kLnRows - 1) / kLnRows), dim3(kLnThreads), 0, stream,
                     static_cast<const _Float16*>(x), static_cast<const _Float16*>(gamma),
                     static_cast<const _Float16*>(beta), static_cast<_Float16*>(y), rows, eps);
  return fw_check_launch("layernorm_rows");
}

extern "C" int fw_gemm_splitk(const void* a, int lda, const void* w, int ldw, float* part, int m, int n, int k,
                              int splits, hipStream_t stream) {
  if (!a || !w || !part) return fw_fail(FW_EINVAL, "gemm_splitk: null pointer");
  if (splits != 2) return fw_fail(FW_EINVAL, "gemm_splitk: splits must be 2");
  if (m <= 0 || n <= 0 || n % kBN || k <= 0 || k % (splits * kBK))
    return fw_fail(FW_EINVAL, "gemm_splitk: need m > 0, n %% %d == 0, k %% %d == 0 (m=%d n=%d k=%d)", kBN,
                   splits * kBK, m, n, k);
  if (lda < k || ldw < k || lda % 8 || ldw % 8 || !aligned16(a) || !aligned16(w) || !aligned16(part))
    return fw_fail(FW_EINVAL, "gemm_splitk: leading dimensions must cover k and be multiples of 8; 16-byte aligned");
  GemmArgs g{};
  g.a = static_cast<const _Float16*>(a);
  g.lda = lda;
  g.w = static_cast<const _Float16*>(w);
  g.ldw = ldw;
  g.m = m;
  g.n = n;
  g.k = k / splits;  // per split
  g.splits = splits;
  g.part = part;
  if (!copy_offsets_fit(g)) return fw_fail(FW_EINVAL, "gemm_splitk: each operand must span less than 4 GiB");
  switch (choose_tile(g, [](Tile t) { return t == kD128 || (t > kD64 && t != kWide256); })) {
    case kS96x64: return launch_ks_partial<96, 64>(g, stream);
    case kS64x64: return launch_ks_partial<64, 64>(g, stream);
    case kS64x32: return launch_ks_partial<64, 32>(g, stream);
    case kS32x32: return launch_ks_partial<32, 32>(g, stream);
    default: break;
  }
  // the XCD rectangles of the plain GEMMs (both k halves of a tile land on the same XCD when the tile
  // count is a multiple of 8): 126 -> 84 MB fetched from beyond L2 for the encoder's fc2
  choose_xcd_groups(g, 128);
  const int tiles = (n / kBN) * ((m + 127) / 128);
  hipLaunchKernelGGL((gemm_dma_kernel<128, kEpiPartial>), dim3(splits * tiles), dim3(gemm_waves<128>() * 64), 0,
                     stream, FW_GEMM_ARGS(g));
  return fw_check_launch("gemm_splitk");
}

extern "C" int fw_layernorm_rows_residual(const float* part, int splits, const void* bias, void* h,
                                          const void* gamma, const void* beta, void* y, int rows, int n, float eps,
                                          int epilogue, hipStream_t stream) {
  if (!part || !bias || !h || !gamma || !beta || !y) return fw_fail(FW_EINVAL, "layernorm_rows_residual: null pointer");
  if (splits != 2) return fw_fail(FW_EINVAL, "layernorm_rows_residual: splits must be 2");
  if (n != kHidden || rows <= 0) return fw_fail(FW_EINVAL, "layernorm_rows_residual: n must be %d", kHidden);
  if (epilogue != FW_EPI_BIAS_RESID && epilogue != FW_EPI_BIAS_RESID_CLAMP)
    return fw_fail(FW_EINVAL, "layernorm_rows_residual: epilogue must be a residual epilogue");
  if (!aligned16(part) || !aligned16(bias) || !aligned16(h) || !aligned16(gamma) || !aligned16(beta) || !aligned16(y))
    return fw_fail(FW_EINVAL, "layernorm_rows_residual: tensors must be 16-byte aligned");
  const dim3 grid((rows + kLnRows - 1) / kLnRows);
  if (epilogue == FW_EPI_BIAS_RESID_CLAMP)
    hipLaunchKernelGGL(residual_layernorm_rows_kernel<true>, grid, dim3(kLnThreads), 0, stream, part,
                       static_cast<const _Float16*>(bias), static_cast<_Float16*>(h),
                       static_cast<const _Float16*>(gamma), static_cast<const _Float16*>(beta),
                       static_cast<_Float16*>(y), rows, eps);
  else
    hipLaunchKernelGGL(residual_layernorm_rows_kernel<false>, grid, dim3(kLnThreads), 0, stream, part,
                       static_cast<const _Float16*>(bias), static_cast<_Float16*>(h),
                       static_cast<const _Float16*>(gamma), static_cast<const _Float16*>(beta),
                       static_cast<_Float16*>(y), rows, eps);
  return fw_check_launch("layernorm_rows_residual");
}


extern "C" int fw_encoder_qkv(const void* y, const void* w, const void* bias, void* qkv, void* vt, int seq, int heads,
                              hipStream_t stream) {
  if (!y || !w || !qkv || !vt) return fw_fail(FW_EINVAL, "encoder_qkv: null pointer");
  const int d = heads * kHeadDim;
  if (seq <= 0 || heads <= 0 || d % kBN || d % kBK)
    return fw_fail(FW_EINVAL, "encoder_qkv: need seq > 0 and heads * 64 a multiple of %d (seq=%d heads=%d)", kBN, seq,
                   heads);
  if (!aligned16(y) || !aligned16(w)) return fw_fail(FW_EINVAL, "encoder_qkv: y and w must be 16-byte aligned");
  if (reinterpret_cast<uintptr_t>(vt) & 7u) return fw_fail(FW_EINVAL, "encoder_qkv: vt must be 8-byte aligned");
  GemmArgs g{static_cast<const _Float16*>(y), d, static_cast<const _Float16*>(w), d,
             static_cast<const _Float16*>(bias), static_cast<_Float16*>(qkv), 3 * d, nullptr, 0, seq, 3 * d, d, d,
             0, 0, 0, heads, seq, static_cast<_Float16*>(vt), vt_pad(seq)};
  return launch_gemm(g, kEpiQkvVt, stream);
}



extern "C" int fw_cross_kv(const void* enc, int t, const void* w, const void* bias, void* cross_kv, int layers,
                           int heads, hipStream_t stream) {
  if (!enc || !w || !cross_kv) return fw_fail(FW_EINVAL, "cross_kv: null pointer");
  if (t <= 0 || layers <= 0 || heads * kHeadDim != kHidden)
    return fw_fail(FW_EINVAL, "cross_kv: need t > 0, layers > 0, heads * 64 == %d", kHidden);
  if (!aligned16(enc) || !aligned16(w) || !aligned8(cross_kv) || (bias && !aligned8(bias)))
    return fw_fail(FW_EINVAL, "cross_kv: enc and w must be 16-byte aligned, cross_kv and bias 8-byte aligned");
  const int n = layers * 2 * kHidden;
  GemmArgs g{static_cast<const _Float16*>(enc), kHidden, static_cast<const _Float16*>(w), kHidden,
             static_cast<const _Float16*>(bias), static_cast<_Float16*>(cross_kv), 0, nullptr, 0, t, n, kHidden, 0,
             0, 0, 0, heads, t};
  return launch_gemm(g, kEpiCrossKV, stream);
}
