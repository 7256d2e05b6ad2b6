// Whisper encoder self-attention for gfx950 (transformers models/whisper/modeling_whisper.py:284-358,
// SDPA path, fp16 in and out, fp32 softmax and accumulation), plus the transposed-V packing it reads.
// Built with MFMA results in VGPRs (-mllvm -amdgpu-mfma-vgpr-form): the softmax reads every score and
// the O accumulators are rescaled in place, which in the AGPR form costs a register move per value.
#include <type_traits>
#include "lds_pipe.h"

namespace fw {
namespace {

// ------------------------------------------------------------------------------------------
// Encoder self-attention, flash style, non-causal, scale 1 (q is pre-scaled by the projection).
// Block = (head, 32 QG queries), 8 waves: QG query groups of 32 x KP key parts (64-key tiles t with
// t % KP == part), so two waves share each SIMD and one's softmax overlaps the other's MFMAs; the parts'
// (m, l, O) are merged through LDS at the end. All waves share one LDS ring whose stages hold KP tiles.
// Per tile a wave computes S^T = K Q^T (keys x queries) with MFMA, so that every lane holds the scores
// of a single query column and the online-softmax max/sum need one cross-lane step (lane ^ 32).
// P^T is fed straight from the S^T accumulator layout as the B operand of O^T = V^T P^T.
//  - Inputs: q and k from the projection output qkv[seq, 3 * heads * 64]; V from a transposed copy
//    vt[heads][64][seq_pad] written by the projection's epilogue, whose key order inside every
//    16-key group has bits 2 and 3 of the key index swapped. With that order the 8 keys an MFMA
//    A-operand lane needs for V^T are one contiguous 16-byte chunk, and they are the keys the
//    same lane holds for P^T in the S^T accumulator (rows 8 (r / 4) + 4 g + (r % 4)).
//  - K tiles (64 keys x 128 B) and V^T tiles (64 d x 128 B) arrive by direct-to-LDS copies into a
//    ring of ST stages, XOR-swizzled by 16-byte chunk like the GEMM tiles.
//  - Block ids are remapped so that the query blocks of a head run on one XCD and its K/V stay in
//    that XCD's L2.
// What bounds it: per tile and wave 16 MFMAs (512 clocks of its SIMD) and about 130 vector instructions,
// 32 of them exponentials (about 700 clocks); two waves share the SIMD, and their phases overlap only in
// part (1.2 us a stage on an idle chip, 1.4 us with every CU busy; leaving out the exponentials, the PV
// products, the copies or the LDS reads gains 0.05 to 0.2 us each).
// EARLY: a tile's operands are in registers before they are needed. V^T is requested behind its first
// score products, and once it has arrived the stage's one barrier frees the stage, so the next tile's K
// is read while this one's softmax runs and a ring of two stages suffices. With four stages reading
// them as the MFMAs take them is as fast (20.6 against 20.9 us for 1500 x 20) and takes 130 registers
// instead of 172.
// ------------------------------------------------------------------------------------------
constexpr int kEaWaves = 8, kEaKV = 64;
constexpr int kEaTileBytes = kEaKV * 128;  // one K tile or one V^T tile

// The QG waves of a key part fill one tile (K then V^T) of a ring stage; `wave` is the wave's query group.
template <int QG>
__device__ __forceinline__ void ea_dma(const _Float16* kbase, int ld, const _Float16* vtbase, int seq_pad,
                                       int seq, int kv0, int wave, int lane, uint32_t stage) {
  constexpr int kN = 8 / QG;  // 8-row blocks per wave of each tile
  const int rsub = lane >> 3, slot = lane & 7;
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    const int blk = kN * wave + i, row = blk * 8 + rsub;
    const int key = min(kv0 + row, seq - 1);  // keys past seq are masked to -inf
    dma16(kbase + static_cast<size_t>(key) * ld + swz_slot(row, slot) * 8,
          __builtin_amdgcn_readfirstlane(stage + blk * 1024));
  }
#pragma unroll
  for (int i = 0; i < kN; ++i) {  // V^T tile: rows are head dims
    const int blk = kN * wave + i, d = blk * 8 + rsub;
    dma16(vtbase + static_cast<size_t>(d) * seq_pad + kv0 + swz_slot(d, slot) * 8,
          __builtin_amdgcn_readfirstlane(stage + kEaTileBytes + blk * 1024));
  }
}

// The same copies for a tile whose 64 keys all lie below seq (every tile but a partial last one): the
// tile's first key only moves the scalar bases, and each lane keeps the byte offsets of its chunks
// (rows of 64 keys or head dims times the row pitch, plus the swizzled chunk), so a stage costs no
// vector address arithmetic. The host keeps 64 rows of either operand within the 32-bit offsets.
template <int QG>
struct EaCopyOffsets {
  uint32_t k[8 / QG], v[8 / QG];
};

template <int QG>
__device__ __forceinline__ EaCopyOffsets<QG> ea_offsets(int ld, int seq_pad, int wave, int lane) {
  const int rsub = lane >> 3, slot = lane & 7;
  EaCopyOffsets<QG> o;
#pragma unroll
  for (int i = 0; i < 8 / QG; ++i) {
    const int row = (8 / QG * wave + i) * 8 + rsub;  // key row of the K tile, head dim of the V^T tile
    o.k[i] = static_cast<uint32_t>((row * ld + swz_slot(row, slot) * 8) * 2);
    o.v[i] = static_cast<uint32_t>((row * seq_pad + swz_slot(row, slot) * 8) * 2);
  }
  return o;
}

template <int QG>
__device__ __forceinline__ void ea_dma_full(const _Float16* kbase, int ld, const _Float16* vtbase, int kv0,
                                            const EaCopyOffsets<QG>& o, int wave, uint32_t stage) {
  constexpr int kN = 8 / QG;
  const _Float16* kb = kbase + static_cast<size_t>(kv0) * ld;
  const _Float16* vb = vtbase + kv0;
#pragma unroll
  for (int i = 0; i < kN; ++i) dma16_s(o.k[i], kb, stage + (kN * wave + i) * 1024);
#pragma unroll
  for (int i = 0; i < kN; ++i) dma16_s(o.v[i], vb, stage + kEaTileBytes + (kN * wave + i) * 1024);
}

// Scores are kept in log2 units (x log2 e). The running max m used for p = exp2(s - m) is only moved
// when some lane of the wave sees a score more than kEaSlack above it, so p stays in [0, 2^kEaSlack]
// (exact in fp16's range) and the O/l rescale runs on few tiles instead of every tile.
constexpr float kEaSlack = 8.f;
constexpr float kLog2e = 1.4426950408889634f;

struct EaState {
  f16v o[2];  // O^T blocks: d in [0, 32) and [32, 64)
  float m, l;
};

// A tile's MFMA operands: K rows 32 b + lane % 32, k-step k of 16 head dims; V^T rows 32 db + lane % 32,
// 16-key step j.
struct EaFrags {
  h8v f[2][4];
};
__device__ __forceinline__ void ea_read(const u32x4* t, int lr, int lg, EaFrags& f) {
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int b = 0; b < 2; ++b) f.f[b][k] = __builtin_bit_cast(h8v, t[swz(32 * b + lr, 2 * k + lg)]);
}

// S^T = K Q^T for two 32-key blocks, their two chains of MFMAs interleaved. V^T of the tile is requested
// behind the first pair: K has arrived by then, so nothing waits for both, and the other MFMAs cover it.
__device__ __forceinline__ void ea_scores(const EaFrags& kf, const h8v (&qf)[4], f16v (&s)[2], const u32x4* vtt, int lr,
                                          int lg, EaFrags& vf) {
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[b][r] = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
#pragma unroll
    for (int b = 0; b < 2; ++b) s[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf.f[b][k], qf[k], s[b], 0, 0, 0);
    if (k == 0) {
      __builtin_amdgcn_sched_barrier(0);
      ea_read(vtt, lr, lg, vf);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// `v(db, j)` gives the V^T operand of head dims 32 db .. and 16-key step j.
template <bool kMask, class V>
__device__ __forceinline__ void ea_softmax_pv(f16v (&s)[2], V v, int kv0, int seq, int lg, EaState& st) {
  float tmax = -INFINITY;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if constexpr (kMask) {
        if (kv0 + 32 * b + 8 * (r >> 2) + 4 * lg + (r & 3) >= seq) s[b][r] = -INFINITY;
      }
      tmax = fmaxf(tmax, s[b][r]);
    }
  tmax = xor_max<32>(tmax) * kLog2e;
  if (__builtin_amdgcn_ballot_w64(tmax > st.m + kEaSlack)) {  // wave-uniform
    const float m_new = fmaxf(st.m, tmax);
    const float corr = __builtin_amdgcn_exp2f(st.m - m_new);  // 0 on the first tile (m = -inf)
    st.l *= corr;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) st.o[b][r] *= corr;
    st.m = m_new;
  }
  float psum = 0.f;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    h8v pf[2];  // P^T of this 32-key block as B operand, [k-step of 16 keys]
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      h2v ph;
      ph[0] = f2h(__builtin_amdgcn_exp2f(fmaf(s[b][r], kLog2e, -st.m)));
      ph[1] = f2h(__builtin_amdgcn_exp2f(fmaf(s[b][r + 1], kLog2e, -st.m)));
      psum = __builtin_amdgcn_fdot2(ph, h2v{static_cast<_Float16>(1.f), static_cast<_Float16>(1.f)}, psum, false);
      pf[r >> 3][r & 7] = ph[0];
      pf[r >> 3][(r & 7) + 1] = ph[1];
    }
    // O^T[d][q] += sum_keys V^T[d][key] P^T[key][q]; k-step (b, hs) covers keys 32 b + 16 hs + [0, 16),
    // whose transposed-layout chunk for lane half lg is chunk 4 b + 2 hs + lg of the V^T row.
#pragma unroll
    for (int hs = 0; hs < 2; ++hs)
#pragma unroll
      for (int db = 0; db < 2; ++db)
        st.o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v(db, 2 * b + hs), pf[hs], st.o[db], 0, 0, 0);
  }
  st.l += xor_add<32>(psum);
}

template <int QG, int KP, int ST, bool EARLY>
__global__ void __launch_bounds__(kEaWaves * 64) encoder_attention_kernel(const _Float16* __restrict__ qkv,
                                                                         const _Float16* __restrict__ vt,
                                                                         _Float16* __restrict__ out, int seq,
                                                                         int heads) {
  static_assert(QG * KP == kEaWaves && 8 % QG == 0, "wave layout");
  constexpr int kPerStage = 2 * 8 / QG;                // copies per thread per stage
  constexpr int kStageBytes = KP * 2 * kEaTileBytes;   // K + V^T of KP tiles
  constexpr int kQ = 32 * QG, kMergeF = 34;            // queries per block; floats per lane of a merged part
  __shared__ __align__(1024) u32x4 ring[ST * kStageBytes / 16];
  static_assert(ST * kStageBytes >= (KP - 1) * QG * 64 * kMergeF * 4, "merge buffer fits in the ring");

  const int qblocks = (seq + kQ - 1) / kQ, nblk = qblocks * heads;
  const int bid = blockIdx.x, full = (nblk / 8) * 8;
  const int job = bid < full ? (bid % 8) * (full / 8) + bid / 8 : bid;
  const int head = job / qblocks, qb = job % qblocks;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wq = wave % QG, part = wave / QG;  // query group, key part (both wave-uniform)
  const int lr = lane & 31, lg = lane >> 5;
  const int ld = 3 * heads * kHeadDim, seq_pad = vt_pad(seq);
  const int q_row = qb * kQ + wq * 32 + lr;  // this lane's query column
  const _Float16* kbase = qkv + (heads + head) * kHeadDim;
  const _Float16* vtbase = vt + static_cast<size_t>(head) * kHeadDim * seq_pad;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(ring));

  // Q^T as B operand: lane holds Q[q_row][16 s + 8 lg .. + 7] for s = 0..3.
  h8v qf[4];
  {
    const _Float16* qp = qkv + static_cast<size_t>(min(q_row, seq - 1)) * ld + head * kHeadDim + 8 * lg;
#pragma unroll
    for (int k = 0; k < 4; ++k) qf[k] = *reinterpret_cast<const h8v*>(qp + 16 * k);
  }
  const int nt = seq_pad / kEaKV, nst = (nt + KP - 1) / KP;
  // Stage p holds tiles KP p .. KP p + KP - 1. A part whose tile is past the end copies the last tile
  // again, so every thread issues the same number of copies per stage (the vmcnt waits count this
  // thread's own copies).
  const EaCopyOffsets<QG> co = ea_offsets<QG>(ld, seq_pad, wq, lane);
  auto issue = [&](int p) {
    const int t = min(KP * p + part, nt - 1);
    const uint32_t stage = lds0 + (p % ST) * kStageBytes + part * 2 * kEaTileBytes;
    if ((t + 1) * kEaKV <= seq)  // wave-uniform; both forms issue the same copies
      ea_dma_full<QG>(kbase, ld, vtbase, t * kEaKV, co, wq, stage);
    else
      ea_dma<QG>(kbase, ld, vtbase, seq_pad, seq, t * kEaKV, wq, lane, stage);
  };
#pragma unroll
  for (int k = 0; k < ST; ++k)
    if (k < nst) issue(k);

  EaState st;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) st.o[b][r] = 0.f;
  st.m = -INFINITY;
  st.l = 0.f;

  auto tile = [&](int p) { return ring + ((p % ST) * kStageBytes + part * 2 * kEaTileBytes) / 16; };  // K, then V^T
  if constexpr (EARLY) {
    EaFrags kf, vf;
    auto v = [&](int db, int j) { return vf.f[db][j]; };
    wait_stages_ahead<kPerStage, ST - 1>(min(ST - 1, nst - 1));
    barrier_only();
    ea_read(tile(0), lr, lg, kf);
    for (int p = 0; p < nst - 1; ++p) {  // every tile of these stages is full
      f16v s[2];
      ea_scores(kf, qf, s, tile(p) + kEaTileBytes / 16, lr, lg, vf);
      // this thread's copies of stage p + 1 have landed, and its own reads of stage p are done: past the
      // barrier the stage is visible to every wave and stage p's slot is free
      wait_stages_ahead<kPerStage, ST - 1>(min(ST - 2, nst - 2 - p));
      lds_barrier();
      if (p + ST < nst) issue(p + ST);
      ea_read(tile(p + 1), lr, lg, kf);
      __builtin_amdgcn_sched_barrier(0);
      ea_softmax_pv<false>(s, v, 0, seq, lg, st);
    }
    const int last = KP * (nst - 1) + part;  // this wave's tile of the last stage, if there is one
    if (last < nt) {
      f16v s[2];
      ea_scores(kf, qf, s, tile(nst - 1) + kEaTileBytes / 16, lr, lg, vf);
      if ((last + 1) * kEaKV <= seq)
        ea_softmax_pv<false>(s, v, last * kEaKV, seq, lg, st);
      else
        ea_softmax_pv<true>(s, v, last * kEaKV, seq, lg, st);
    }
  } else {
    auto step = [&](auto mask, int p) {  // this wave's tile of stage p, operands read as the MFMAs take them
      const u32x4* kt = tile(p);
      auto v = [&](int db, int j) {
        return __builtin_bit_cast(h8v, kt[kEaTileBytes / 16 + swz(32 * db + lr, 2 * j + lg)]);
      };
      f16v s[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[b][r] = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const h8v kv = __builtin_bit_cast(h8v, kt[swz(32 * b + lr, 2 * k + lg)]);
          s[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kv, qf[k], s[b], 0, 0, 0);
        }
      }
      ea_softmax_pv<decltype(mask)::value>(s, v, (KP * p + part) * kEaKV, seq, lg, st);
    };
    auto next = [&](int p) {  // stage p visible to every wave; every wave is done with stage p - 1
      wait_stages_ahead<kPerStage, ST - 1>(min(p ? ST - 2 : ST - 1, nst - 1 - p));
      barrier_only();
      if (p > 0 && p + ST - 1 < nst) issue(p + ST - 1);
    };
    for (int p = 0; p < nst - 1; ++p) {  // every tile of these stages is full
      next(p);
      step(std::false_type{}, p);
    }
    next(nst - 1);
    const int last = KP * (nst - 1) + part;
    if (last < nt) {
      if ((last + 1) * kEaKV <= seq)
        step(std::false_type{}, nst - 1);
      else
        step(std::true_type{}, nst - 1);
    }
  }

  // Merge the key parts: parts 1 .. KP - 1 hand (m, l, O) through LDS to the wave of part 0 with the same
  // query group; lane for lane the registers describe the same query and head dims.
  lds_barrier();  // every wave is done with the ring
  float* mbuf = reinterpret_cast<float*>(ring) + (wq * 64 + lane) * kMergeF;
  constexpr int kPartF = QG * 64 * kMergeF;  // floats of one part
  if (part > 0) {
    float* mine = mbuf + (part - 1) * kPartF;
    mine[0] = st.m;
    mine[1] = st.l;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[2 + 16 * b + r] = st.o[b][r];
  }
  lds_barrier();
  if (part > 0 || q_row >= seq) return;
  float m = st.m, a[KP];  // a part without a tile has m = -inf, l = 0
#pragma unroll
  for (int i = 1; i < KP; ++i) m = fmaxf(m, mbuf[(i - 1) * kPartF]);
  a[0] = __builtin_amdgcn_exp2f(st.m - m);
  float l = st.l * a[0];
#pragma unroll
  for (int i = 1; i < KP; ++i) {
    a[i] = __builtin_amdgcn_exp2f(mbuf[(i - 1) * kPartF] - m);
    l += mbuf[(i - 1) * kPartF + 1] * a[i];
  }
  const float inv = 1.0f / l;
  _Float16* orow = out + static_cast<size_t>(q_row) * heads * kHeadDim + head * kHeadDim;
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      h4v v4;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * j + e;
        float o = st.o[db][r] * a[0];
#pragma unroll
        for (int i = 1; i < KP; ++i) o += mbuf[(i - 1) * kPartF + 2 + 16 * db + r] * a[i];
        v4[e] = f2h(o * inv);
      }
      *reinterpret_cast<h4v*>(orow + 32 * db + 8 * j + 4 * lg) = v4;
    }
}

// Transposed V for the attention kernel from a projection output (qkv v columns).
__global__ void __launch_bounds__(256) pack_vt_kernel(const _Float16* __restrict__ qkv, _Float16* __restrict__ vt,
                                                      int seq, int heads) {
  const int seq_pad = vt_pad(seq);
  const int i = blockIdx.x * 256 + threadIdx.x;  // over heads * 64 * seq_pad
  if (i >= heads * kHeadDim * seq_pad) return;
  const int pos = i % seq_pad, hd = i / seq_pad;  // hd = head * 64 + d
  const int t = vt_pos(pos);
  vt[i] = t < seq ? qkv[static_cast<size_t>(t) * 3 * heads * kHeadDim + 2 * heads * kHeadDim + hd]
                  : static_cast<_Float16>(0.f);
}


bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

}  // namespace
}  // namespace fw

using namespace fw;

extern "C" long long fw_encoder_vt_elems(int seq, int heads) {
  if (seq <= 0 || heads <= 0) return 0;
  return static_cast<long long>(heads) * kHeadDim * vt_pad(seq);
}

extern "C" int fw_encoder_pack_vt(const void* qkv, void* vt, int seq, int heads, hipStream_t stream) {
  if (!qkv || !vt) return fw_fail(FW_EINVAL, "encoder_pack_vt: null pointer");
  if (seq <= 0 || heads <= 0) return fw_fail(FW_EINVAL, "encoder_pack_vt: seq and heads must be positive");
  const long long n = fw_encoder_vt_elems(seq, heads);
  hipLaunchKernelGGL(pack_vt_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, stream,
                     static_cast<const _Float16*>(qkv), static_cast<_Float16*>(vt), seq, heads);
  return fw_check_launch("encoder_pack_vt");
}

extern "C" int fw_encoder_attention(const void* qkv, const void* vt, void* out, int seq, int heads,
                                    hipStream_t stream) {
  if (!qkv || !vt || !out) return fw_fail(FW_EINVAL, "encoder_attention: null pointer");
  if (seq <= 0 || heads <= 0) return fw_fail(FW_EINVAL, "encoder_attention: seq and heads must be positive");
  // 64 rows of K (pitch 3 heads 64) or of V^T (pitch vt_pad(seq)) within the copies' 32-bit byte offsets
  if (64LL * 3 * heads * kHeadDim * 2 >= (1LL << 32) || 64LL * vt_pad(seq) * 2 >= (1LL << 32))
    return fw_fail(FW_EINVAL, "encoder_attention: seq or heads too large");
  if (!aligned(qkv, 16) || !aligned(vt, 16) || !aligned(out, 8))
    return fw_fail(FW_EINVAL, "encoder_attention: qkv and vt must be 16-byte aligned, out 8-byte aligned");
  const auto launch = [&](auto kernel, int queries) {
    hipLaunchKernelGGL(kernel, dim3((seq + queries - 1) / queries * heads), dim3(kEaWaves * 64), 0, stream,
                       static_cast<const _Float16*>(qkv), static_cast<const _Float16*>(vt),
                       static_cast<_Float16*>(out), seq, heads);
  };
  // 128 queries a block, so that each K/V tile is staged once for all of them, while that gives more than
  // half the CUs a block; otherwise 64 queries and four key parts: twice the blocks, each with half the
  // chain of tiles (20 heads, us by 128 / 64 queries: 251 keys 7.1 / 6.1, 640 keys 10.6 / 8.2, 768 keys
  // 12.1 / 9.4, 1000 keys 14.5 / 19.3). With at most two tiles there is no chain to shorten (64 keys 4.1 / 5.2).
  if ((seq + 127) / 128 * heads > 128 || seq <= 2 * kEaKV)
    launch(encoder_attention_kernel<4, 2, 4, false>, 128);
  else
    launch(encoder_attention_kernel<2, 4, 2, true>, 64);
  return fw_check_launch("encoder_attention");
}
