// Joint-attention forward on gfx950: O = softmax(Q K^T * scale) V per head,
// non-causal, no mask, bf16 in / bf16 out, fp32 softmax and accumulation, head
// dim 128 -- the reference model's F.scaled_dot_product_attention(q, k, v,
// is_causal=False) (deploy/xvideo/models/dit/dit.py:154-167), which the block
// calls on the joint Q = [video | condition] and K, V = [cached | video |
// condition] (dit.py:489-498).
//
// Layout: Q, K, V and O are token-major [L, H, 128] views (token and head strides
// in elements), so the joint operands are read where the fused QKV / pack ops wrote
// them and O is written straight into the [L, H*128] rows the out-projection reads.
//
// One wave = 32 queries of one head, 8 waves per workgroup (one workgroup per CU), one pass over
// the keys in tiles of 64 (flash attention with an online softmax), each tile as two 32-key
// halves with a softmax step each. Per half and wave:
//   * S^T = K Q^T: 8 v_mfma_f32_32x32x16_bf16 (K from LDS as the A operand, the wave's 32
//     queries kept in registers as the B operand). In the 32x32 output a lane holds 16 keys of
//     ONE query, so the row max / row sum are in-lane plus one exchange with lane ^ 32;
//   * online softmax in fp32 with exp2 (scale * log2 e folded into the scores), computed first
//     against the running max and redone with the half's row max only when a probability could
//     reach 2^7 (the first tile, or scores well above the running max);
//   * O^T += V^T P^T: 8 MFMAs; P^T is the B operand straight from the registers that hold the
//     scores (rounded to bf16), which fixes a permutation of the 16 keys of each MFMA; the A
//     operand (V^T) comes from the key-major V tile with two ds_read_b64_tr_b16 per MFMA, whose
//     addresses apply the same permutation. The O^T accumulator again gives each lane one
//     query, so the rescale by exp2(m_old - m_new) is per lane.
// The two halves are software-pipelined inside the wave: S(0); S(1) with the softmax of half 0
// on the VALU; PV(0) with the softmax of half 1; PV(1). The A operands of the tile's 32 MFMAs
// (K, then the transposed V) are fetched from LDS two MFMAs ahead of their use.
// K and V tiles reach LDS by buffer DMA straight into LDS (double-buffered, the next tile in
// flight during the current one, one barrier per tile); LDS rows of 256 bytes store 16-byte
// chunk c at a row-dependent XOR of c (chunk_at, chunk_at_v).
//
// ds_read_b64_tr_b16 lane layout (measured on gfx950): within each group of 16
// lanes, lane a points at 4 consecutive 16-bit values M[a][0..3] and lane i receives
// M[4j + i/4][i % 4] for j = 0..3.
#include <cfloat>
#include <type_traits>

#include "joy_common.hpp"
#include "joy_kernels.hpp"

namespace joy {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kD = 128;
constexpr int kBK = 64;                // keys per tile
constexpr int kRowB = kD * 2;          // bytes per K / V row
constexpr int kTileB = kBK * kRowB;    // 16 KB per K or V tile

template <int J>
using IC = std::integral_constant<int, J>;

// K tile: 16-byte chunk c of key row r at c ^ (r & 15) -- the fragment reads take 16 consecutive rows of one
// logical chunk. V tile: c ^ vsw(r) -- a transpose read takes rows 4n..4n+3 and logical chunks 4m..4m+3
// (32 lanes), which vsw spreads over 16 distinct physical chunks (and over 8 distinct chunk positions mod 8 per
// 16 lanes), where (r & 15) folded them onto 4.
__device__ __forceinline__ int chunk_at(int row, int chunk) { return row * kRowB + ((chunk ^ (row & 15)) << 4); }
__device__ __forceinline__ int vsw(int row) { return ((row & 1) << 2) ^ ((row & 2) ? 10 : 0); }
__device__ __forceinline__ int chunk_at_v(int row, int chunk) { return row * kRowB + ((chunk ^ vsw(row)) << 4); }

__device__ __forceinline__ v16f mfma_bf16(const bf16x8& a, const bf16x8& b, const v16f& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 as_bf16x8(const v4i& v) { return __builtin_bit_cast(bf16x8, v); }

// Buffer load of 16 bytes per lane (offset voff + soff within the descriptor's range, zeros past
// it) into LDS at m0 = lds_dst (wave-uniform) + lane * 16, as inline asm: the compiler then does
// not track these LDS writes, and the only wait on them is the explicit vmcnt(0) at the top of
// each key tile. (Through the builtin, the compiler cannot tell the transpose reads of the
// current tile from the DMA into the other buffer and waits for the in-flight next tile before
// them.) m0 is written only here in this file, and nothing else in the kernel reads it (checked in
// the generated code): the compiler's warning that a clobber of this reserved register is not
// preserved does not apply.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16_buf(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, int soff, lds_void* lds_dst) {
  const uint32_t m = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds_dst);
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(m), "v"(voff), "s"(rsrc),
               "s"(soff)
               : "m0");
}
#pragma clang diagnostic pop

// Combine a value with the one of lane ^ 32 without the LDS crossbar: v_permlane32_swap
// with both operands x returns {x[lane], x[lane ^ 32]} (in an order that depends on the
// half, measured on gfx950), and both halves add them in the same order.
__device__ __forceinline__ float xor32_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor32_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// One query block of 32 queries per wave, 8 waves per workgroup (one workgroup per CU, two waves
// per SIMD): the workgroup's 256 queries share every K / V tile it moves into LDS, half the DMA
// traffic per query of 128-query workgroups (measured 3.5 % faster at the cfg-4 shape). Each
// 64-key tile is processed as two 32-key halves with an online-softmax step each, so that within
// the wave the VALU work of one half overlaps the MFMAs of the other: S(0); S(1) with
// softmax(0); PV(0) with softmax(1); PV(1). A softmax step follows each MFMA in program order
// (sched_barrier keeps it there).
//
// Work split: the query blocks of all heads form one list (head-major, qb_per_head blocks per
// head) and workgroup w takes blocks 8 w .. 8 w + 7, so the grid has ceil(heads * qb_per_head / 8)
// workgroups whatever the query count per head (per-head workgroups would leave a nearly empty
// last round at 11312 queries: 45 x 40 = 1800 = 7.03 rounds of 256 CUs). A workgroup whose blocks
// straddle a head boundary moves the K / V tiles of both heads (LDS holds two heads' tiles);
// qb_per_head >= 8 keeps it to two heads. Blocks past the list (last workgroup) compute on the
// last valid block and store nothing.
//
// Key split (AttnSplit, split_plan): the groups past the last whole round of the chip can be cut
// along the keys, a part per workgroup. A part leaves its unnormalised fp32 O and its running max
// and sum in the workspace, and attn_combine adds a group's parts in key order. A workgroup takes
// one part only: a loop over several in one workgroup costs 114 VGPR spills. What the kernel is
// bound by stays as above (LDS operand reads and power); the split fills idle CUs. Measured against
// the unsplit call, the second launch included: 512 x 8000 x 32 heads 183 -> 73 us, 859 x 5000 x 32 132 -> 95,
// 5000 x 5000 x 40 554 -> 472, 3467 x 11267 x 32 626 -> 603. (wave is moved to a scalar register, so that the DMA's
// LDS addresses are scalars: 250 -> 248 VGPRs with the split's code, 0.5-3 % faster unsplit.)
constexpr int kWaves = 8;
constexpr int kPartBlock = 64 * 64 + 64;        // floats per query block of a part: O, then m and l of 32 queries
constexpr int kPartSlot = kWaves * kPartBlock;  // floats per part (one group)
constexpr int kSplitMinTiles = 4;               // key tiles of a part: below, its prologue and epilogue dominate
struct AttnSplit {
  float* ws;         // [split_groups][parts] slots
  int full_groups;   // the workgroups before the split ones: a whole group each
  int split_groups;
  int parts;         // parts per split group
  int part_tiles;    // key tiles of each part but the last, which has what is left
};

// kSplit: whether the call has split groups. A call without any runs a kernel without their indexing, which
// costs short calls up to 5 % (32 heads: 128 x 128 8.2 against 8.0 us, 347 x 347 18.2 against 17.3, 1371 x 1371 44.5
// against 44.2; from 512 x 512 on mostly level).
template <bool kSplit>
__device__ __forceinline__ void attn_body(const AttnArgs& a, int qb_per_head, const AttnSplit& sp) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[2][2][2][kTileB];  // [buffer][head slot][K, V]
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ql = lane & 31, hf = lane >> 5;
  const int64_t Lq = a.q_len, Lk = a.k_len;
  const int nblocks = a.heads * qb_per_head;
  // this workgroup's group of query blocks and its key tiles [t0, t1)
  const int64_t ntiles = (Lk + kBK - 1) / kBK;
  int group = (int)blockIdx.x;
  int slot = -1;
  int64_t t0 = 0, t1 = ntiles;
  if (kSplit && group >= sp.full_groups) {
    const int w = group - sp.full_groups;
    // part 0 of every group first, then part 1, ... (the shorter last ones at the end); the quotient
    // is uniform but computed on the VALU, so it is moved to a scalar register
    const int part = __builtin_amdgcn_readfirstlane(w / sp.split_groups), g = w - part * sp.split_groups;
    group = sp.full_groups + g;
    slot = g * sp.parts + part;
    t0 = (int64_t)part * sp.part_tiles;
    t1 = min(ntiles, t0 + sp.part_tiles);
  }
  const int blk0 = group * kWaves;
  const int head_lo = __builtin_amdgcn_readfirstlane(blk0 / qb_per_head);
  const int head_hi = __builtin_amdgcn_readfirstlane((min(blk0 + kWaves, nblocks) - 1) / qb_per_head);  // blk0 < nblocks
  const bool straddle = head_hi != head_lo;
  const int blk = min(blk0 + wave, nblocks - 1);
  const bool active = blk0 + wave < nblocks;
  const int head = blk / qb_per_head;
  const int hslot = head == head_lo ? 0 : 1;
  const int qrow = (blk - head * qb_per_head) * 32 + ql;

  v4i qf[8];
  {
    const uint16_t* qp = a.q.ptr + (int64_t)min((int64_t)qrow, Lq - 1) * a.q.stride_token +
                         (int64_t)head * a.q.stride_head + 8 * hf;
#pragma unroll
    for (int st = 0; st < 8; ++st) qf[st] = *(const v4i*)(qp + 16 * st);
  }

  // K / V tiles by buffer DMA: wave w moves rows 8 w .. 8 w + 7 of each (two DMAs of 4 rows), for
  // the workgroup's first head and, when it straddles a head boundary, its second head.
  // The buffer descriptors are rebuilt per tile, based at the tile's first key and ending after
  // its last key below Lk: rows past Lk load zeros (their scores are -inf), and the offsets stay
  // below 64 rows whatever the sequence length.
  const int64_t ks = a.k.stride_token, vs = a.v.stride_token;
  auto dma_head = [&](int buf, int slot, int h, int64_t k0) {
    const uint16_t* kb = a.k.ptr + (int64_t)h * a.k.stride_head;
    const uint16_t* vb = a.v.ptr + (int64_t)h * a.v.stride_head;
    const int rows = (int)min((int64_t)kBK, Lk - k0);
    const __amdgpu_buffer_rsrc_t krs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(kb + k0 * ks), 0, (int)(((rows - 1) * ks + kD) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(vb + k0 * vs), 0, (int)(((rows - 1) * vs + kD) * 2), 0x00020000);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = wave * 8 + i * 4 + (lane >> 4);
      dma16_buf(krs, (uint32_t)(row * ks * 2 + ((lane & 15) ^ (row & 15)) * 16), 0,
                (lds_void*)&lds[buf][slot][0][(wave * 8 + i * 4) * kRowB]);
      dma16_buf(vrs, (uint32_t)(row * vs * 2 + ((lane & 15) ^ vsw(row)) * 16), 0,
                (lds_void*)&lds[buf][slot][1][(wave * 8 + i * 4) * kRowB]);
    }
  };
  auto dma_tile = [&](int buf, int64_t k0) {
    dma_head(buf, 0, head_lo, k0);
    if (straddle) dma_head(buf, 1, head_hi, k0);
  };

  const int tg = lane >> 4, ta = lane & 15;
  const int tr_row = 4 * hf + (ta >> 2);
  const int tr_col = 16 * (tg & 1) + 4 * (ta & 3);

  v16f o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) o[db] = (v16f){};
  float m_run = -INFINITY, l_run = 0.f;
  const float sl2 = a.scale_log2e;

  // Softmax of one 32-key half (16 scores per lane), first against the running max m_run: steps 0-7
  // (one after each MFMA of the phase) compute 2 probabilities each, rounded to a bf16 pair for the
  // PV operand and summed as those bf16 values (v_dot2c_f32_bf16 against (1, 1)), so the row sum
  // normalises exactly the weights the MFMAs apply. The online softmax is exact for any reference
  // point, so the half needs no row max as long as its probabilities stay small: if every lane's sum
  // (16 keys of a query) is below 2^7, every probability is, and the half is done. Else (the first
  // tile, where m_run = -inf, or scores well above m_run) the wave redoes the half against the
  // larger of m_run and its row max (soft_max), and O is rescaled.
  struct Soft {
    float m_new, alpha, rs;
  };
  const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
  // probabilities 2 e and 2 e + 1 against m_ref
  auto probs = [&](int e, const v16f& s, v4i (&pb)[2], float m_ref, float& rs) {
    const float q0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * e], sl2, -m_ref));
    const float q1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * e + 1], sl2, -m_ref));
    const uint32_t pk = pack_bf16x2(q0, q1);
    rs = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pk), one, rs, false);
    pb[e >> 2][e & 3] = (int)pk;
  };
  auto soft_step = [&](int step, const v16f& s, v4i (&pb)[2], Soft& st) {
    if (step == 0) st.rs = 0.f;
    probs(step, s, pb, m_run, st.rs);
  };
  // the same half against max(m_run, row max): its probabilities are then at most 1, and the later
  // halves pass the check unless their scores rise again
  auto soft_max = [&](const v16f& s, v4i (&pb)[2], Soft& st) {
    float m = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) m = fmaxf(fmaxf(m, s[r]), s[r + 1]);
    const float mt = xor32_max(fmaxf(m, s[15]));
    const float m_cand = mt * sl2;
    // finite also where every score so far is -inf, so that such a tile adds nothing instead of NaN
    st.m_new = fmaxf(fmaxf(m_run, m_cand), -FLT_MAX);
    st.alpha = __builtin_amdgcn_exp2f(m_run - st.m_new);
    st.rs = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) probs(e, s, pb, st.m_new, st.rs);
  };
  auto rescale = [&](float alpha) {
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
      for (int db = 0; db < 4; ++db) o[db] *= alpha;
    }
  };
  // Before the half's PV MFMAs: the check, on each lane's 16 keys (a sum below 2^7 there bounds every
  // probability as well), and where it fails the max-based redo and the rescale of O (the rare path,
  // laid out off the fall-through). The row sum over the 32 keys and the running sum follow after the
  // first PV MFMA (soft_sum).
  auto soft_end = [&](const v16f& s, v4i (&pb)[2], Soft& st) {
    st.alpha = 1.0f;
    // false for inf / NaN (m_run = -inf)
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(st.rs < 128.0f)) != 0, 0)) {
      soft_max(s, pb, st);
      m_run = st.m_new;
      rescale(st.alpha);
    }
  };
  auto soft_sum = [&](Soft& st) { l_run = l_run * st.alpha + xor32_sum(st.rs); };
  auto k_operand = [&](const uint8_t* kt, int kb, int st) -> v4i {
    return *(const v4i*)(kt + chunk_at(kb * 32 + ql, 2 * st + hf));
  };
  auto pv_operand = [&](const uint8_t* vt, int kb, int n) -> v4i {  // n = 4 b + db
    const int b = n >> 2, db = n & 3;
    const int row0 = kb * 32 + 16 * b + tr_row;
    const int col = db * 32 + tr_col;
    const int chunk = col >> 3, within = (col & 7) * 2;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vt + chunk_at_v(row0, chunk) + within));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vt + chunk_at_v(row0 + 8, chunk) + within));
    return __builtin_bit_cast(v4i, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  dma_tile(0, t0 * kBK);
  auto tile = [&](auto bufc, auto partc, int64_t t) {
    constexpr int buf = decltype(bufc)::value;
    constexpr bool partial = decltype(partc)::value;
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0), lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (t + 1 < t1) dma_tile(buf ^ 1, (t + 1) * kBK);
    const uint8_t* kt = lds[buf][hslot][0];
    const uint8_t* vt = lds[buf][hslot][1];
    const int64_t k0 = t * kBK;
    auto mask = [&](v16f& s, int kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t key = k0 + kb * 32 + 8 * (r >> 2) + 4 * hf + (r & 3);
        if (key >= Lk) s[r] = -INFINITY;
      }
    };
    v16f s0, s1;
    v4i p0[2], p1[2];
    Soft st0, st1;
    // The tile's 32 MFMAs read one stream of A operands -- K of half 0, K of half 1, V of half 0,
    // V of half 1 -- each fetched from LDS kOperandAhead MFMAs before it is used (one register set
    // per fetch in flight; with the 2 waves per SIMD this hides most of the LDS latency, and at
    // two fetches ahead the kernel still fits 256 registers without spilling).
    constexpr int kOperandAhead = 2;
    constexpr int NB = kOperandAhead + 1;
    v4i ob[NB];
    auto operand = [&](int i) -> v4i {
      if (i < 8) return k_operand(kt, 0, i);
      if (i < 16) return k_operand(kt, 1, i - 8);
      if (i < 24) return pv_operand(vt, 0, i - 16);
      return pv_operand(vt, 1, i - 24);
    };
#pragma unroll
    for (int i = 0; i < NB - 1; ++i) ob[i] = operand(i);
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      if (i + NB - 1 < 32) ob[(i + NB - 1) % NB] = operand(i + NB - 1);
      const v4i op = ob[i % NB];
      if (i < 8) {  // S(0)
        s0 = mfma_bf16(as_bf16x8(op), as_bf16x8(qf[i]), i == 0 ? (v16f){} : s0);
      } else if (i < 16) {  // S(1) with softmax(0)
        s1 = mfma_bf16(as_bf16x8(op), as_bf16x8(qf[i - 8]), i == 8 ? (v16f){} : s1);
        __builtin_amdgcn_sched_barrier(0);
        soft_step(i - 8, s0, p0, st0);
      } else if (i < 24) {  // PV(0) with softmax(1)
        o[(i - 16) & 3] = mfma_bf16(as_bf16x8(op), as_bf16x8(p0[(i - 16) >> 2]), o[(i - 16) & 3]);
        __builtin_amdgcn_sched_barrier(0);
        if (i == 16) soft_sum(st0);
        soft_step(i - 16, s1, p1, st1);
      } else {  // PV(1)
        o[(i - 24) & 3] = mfma_bf16(as_bf16x8(op), as_bf16x8(p1[(i - 24) >> 2]), o[(i - 24) & 3]);
        if (i == 24) {
          __builtin_amdgcn_sched_barrier(0);
          soft_sum(st1);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (i == 7) {
        if constexpr (partial) mask(s0, 0);
        __builtin_amdgcn_sched_barrier(0);
      } else if (i == 15) {
        soft_end(s0, p0, st0);
        if constexpr (partial) mask(s1, 1);
        __builtin_amdgcn_sched_barrier(0);
      } else if (i == 23) {
        soft_end(s1, p1, st1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const int64_t nfull = min(t1, Lk / kBK);
  int64_t t = t0;
  for (; t + 2 <= nfull; t += 2) {
    tile(IC<0>{}, std::false_type{}, t);
    tile(IC<1>{}, std::false_type{}, t + 1);
  }
  if (t < nfull) {
    tile(IC<0>{}, std::false_type{}, t);
    ++t;
    if (t < t1) tile(IC<1>{}, std::true_type{}, t);
  } else if (t < t1) {
    tile(IC<0>{}, std::true_type{}, t);
  }
  __builtin_amdgcn_s_waitcnt(0x0070);

  if (kSplit && slot >= 0) {
    float* pp = sp.ws + (int64_t)slot * kPartSlot + wave * kPartBlock;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        *(float4*)(pp + (db * 4 + r4) * 256 + lane * 4) =
            make_float4(o[db][4 * r4], o[db][4 * r4 + 1], o[db][4 * r4 + 2], o[db][4 * r4 + 3]);
    pp[64 * 64 + lane] = hf == 0 ? m_run : l_run;  // both halves hold their query's m and l
  } else if (active && qrow < Lq) {
    const float inv = 1.0f / l_run;
    uint16_t* op = a.out + (int64_t)qrow * a.out_stride_token + (int64_t)head * kD;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const int d = db * 32 + 8 * r4 + 4 * hf;
        uint2 w;
        w.x = pack_bf16x2(o[db][4 * r4] * inv, o[db][4 * r4 + 1] * inv);
        w.y = pack_bf16x2(o[db][4 * r4 + 2] * inv, o[db][4 * r4 + 3] * inv);
        *(uint2*)(op + d) = w;
      }
  }
}

__global__ __launch_bounds__(64 * kWaves, 1) void attn_fwd_d128(AttnArgs a, int qb_per_head) {
  attn_body<false>(a, qb_per_head, AttnSplit{});
}
__global__ __launch_bounds__(64 * kWaves, 1) void attn_split_d128(AttnArgs a, int qb_per_head, AttnSplit sp) {
  attn_body<true>(a, qb_per_head, sp);
}

// Adds the parts of the split groups in key order: one 256-thread workgroup per query block, wave w
// the 32 output columns of accumulator w of attn_body, in the same lane layout.
__global__ __launch_bounds__(256) void attn_combine(AttnArgs a, int qb_per_head, AttnSplit sp) {
  const int lane = threadIdx.x & 63, db = threadIdx.x >> 6;
  const int ql = lane & 31, hf = lane >> 5;
  const int g = (int)blockIdx.x / kWaves, wave = (int)blockIdx.x % kWaves;
  const int blk = (sp.full_groups + g) * kWaves + wave;
  if (blk >= a.heads * qb_per_head) return;  // padding of the last group
  const int head = blk / qb_per_head;
  const int qrow = (blk - head * qb_per_head) * 32 + ql;
  const float* pp = sp.ws + (int64_t)g * sp.parts * kPartSlot + wave * kPartBlock;
  float4 o[4];
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4) o[r4] = *(const float4*)(pp + (db * 4 + r4) * 256 + lane * 4);
  float m = pp[64 * 64 + ql], l = pp[64 * 64 + 32 + ql];
  for (int p = 1; p < sp.parts; ++p) {
    pp += kPartSlot;
    const float mp = pp[64 * 64 + ql], lp = pp[64 * 64 + 32 + ql];
    const float m_new = fmaxf(m, mp);
    const float sa = __builtin_amdgcn_exp2f(m - m_new), sb = __builtin_amdgcn_exp2f(mp - m_new);
    m = m_new;
    l = l * sa + lp * sb;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const float4 x = *(const float4*)(pp + (db * 4 + r4) * 256 + lane * 4);
      o[r4].x = o[r4].x * sa + x.x * sb;
      o[r4].y = o[r4].y * sa + x.y * sb;
      o[r4].z = o[r4].z * sa + x.z * sb;
      o[r4].w = o[r4].w * sa + x.w * sb;
    }
  }
  if (qrow >= a.q_len) return;
  const float inv = 1.0f / l;
  uint16_t* op = a.out + (int64_t)qrow * a.out_stride_token + (int64_t)head * kD;
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4) {
    uint2 w;
    w.x = pack_bf16x2(o[r4].x * inv, o[r4].y * inv);
    w.y = pack_bf16x2(o[r4].z * inv, o[r4].w * inv);
    *(uint2*)(op + db * 32 + 8 * r4 + 4 * hf) = w;
  }
}

// Key split of the last, partial round: the `rest` groups past the last whole round of the chip
// would take a whole round's time on a part of it. Each is cut into `s` equal parts, s * rest of
// them in one workgroup each at the same time, and one shorter rest; the CUs that the s * rest
// parts leave idle take the rests, at most k = ceil(rest / idle) of them each. With parts of
// k / (1 + k s) of the keys a CU's k rests take as long as one part, so the round ends after that
// share of its time (rest = 180 of 256 CUs: s = 1, k = 3, 3/4; the least any split reaches is
// 180 / 256).
// The split costs the parts' way to memory and back (133 KB each) and a second launch, and the more
// CUs the unsplit round keeps busy, the less it has to give: power sets the clock, so a round on
// part of the chip runs faster per tile. It is taken when it takes at least 5 + 26 rest / cus key
// tiles off the round. Measured (unsplit, split; tiles taken off, rest): 512 x 600 x 32 22.2, 22.1 us
// (8, 64); x 1000 30.4, 24.4 (12, 64); 859 x 859 30.7, 35.8 (8, 108); x 2000 58.6, 50.9 (18, 108);
// 1371 x 2731 78.3, 83.1 (11, 172); x 5000 132, 127 (20, 172); 7367 x 3900 430, 434 (20, 156); x 7367
// 850, 836 (38, 156); 3467 x 3467 208, 214 (14, 180); x 6587 356, 356 (26, 180); 1907 x 12000 357, 369
// (12, 240); x 20000 605, 603 (20, 240).
AttnSplit split_plan(int64_t q_len, int64_t k_len, int heads) {
  const int64_t qb = max((q_len + 31) / 32, (int64_t)kWaves);
  const int64_t groups = (heads * qb + kWaves - 1) / kWaves, ntiles = (k_len + kBK - 1) / kBK;
  const int64_t cus = device_cus(), rest = groups % cus;
  AttnSplit sp = {nullptr, (int)groups, 0, 0, 0};
  if (rest == 0) return sp;
  const int64_t s = cus / rest, idle = cus - s * rest;
  const int64_t k = idle > 0 ? (rest + idle - 1) / idle : 0;
  const int64_t part = max(k > 0 ? (ntiles * k + k * s) / (1 + k * s) : (ntiles + s - 1) / s, (int64_t)kSplitMinTiles);
  const int64_t parts = (ntiles + part - 1) / part;
  if (parts < 2 || (ntiles - part) * cus < 5 * cus + 26 * rest) return sp;
  sp.full_groups = (int)(groups - rest);
  sp.split_groups = (int)rest;
  sp.parts = (int)parts;
  sp.part_tiles = (int)part;
  return sp;
}

}  // namespace

// Tried and dropped (same inputs, cfg-4 joint shape): two query blocks per wave, pipelined inside
// the wave at one wave per SIMD (bit-identical outputs, 9.8 vs 8.2 ms: the scores no longer fit
// the architectural registers and every tile pays accumulator-register copies; rebuilt with two
// waves per workgroup it spills to scratch), and the same kernel without the half-tile split
// (MFMA busy 49 % at 1.94 GHz against 54 % at 1.83 GHz here: the part is power-limited, so the
// better overlap buys 2.6 %). A three-stage K / V ring (next-but-one tile in flight) measured no
// faster than two stages. Two query blocks per wave at one wave per SIMD with the output
// accumulators pinned in a0..a127 by inline asm (no accumulator copies, no spills, bit-identical):
// 3-5 % slower than this kernel -- half the LDS operand reads and a higher clock (2.1 against
// 1.87 GHz), but the single wave's own latencies exposed (MFMA busy 0.47 against 0.55).
int64_t attention_workspace_bytes(int64_t q_len, int64_t k_len, int heads) {
  const AttnSplit sp = split_plan(q_len, k_len, heads);
  return (int64_t)sp.split_groups * sp.parts * kPartSlot * (int64_t)sizeof(float);
}

hipError_t launch_attention_fwd(const AttnArgs& a, void* workspace, int64_t workspace_bytes, hipStream_t st) {
  // query blocks per head: at least kWaves, so a workgroup spans at most two heads
  const int qb = (int)max((a.q_len + 31) / 32, (int64_t)kWaves);
  const int64_t blocks = (int64_t)a.heads * qb;
  AttnSplit sp = split_plan(a.q_len, a.k_len, a.heads);
  if (sp.split_groups > 0 &&
      (!workspace || workspace_bytes < (int64_t)sp.split_groups * sp.parts * kPartSlot * (int64_t)sizeof(float)))
    sp = {nullptr, (int)((blocks + kWaves - 1) / kWaves), 0, 0, 0};
  sp.ws = (float*)workspace;
  if (sp.split_groups == 0) {
    hipLaunchKernelGGL(attn_fwd_d128, dim3((unsigned)sp.full_groups), dim3(64 * kWaves), 0, st, a, qb);
  } else {
    hipLaunchKernelGGL(attn_split_d128, dim3((unsigned)(sp.full_groups + sp.split_groups * sp.parts)),
                       dim3(64 * kWaves), 0, st, a, qb, sp);
    hipLaunchKernelGGL(attn_combine, dim3((unsigned)(sp.split_groups * kWaves)), dim3(256), 0, st, a, qb, sp);
  }
  return hipGetLastError();
}

}  // namespace joy
