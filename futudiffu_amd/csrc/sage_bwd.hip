// Sage attention backward for gfx950 (CDNA4).
//
// Reference: the Triton kernels of sqcu/futudiffu src/futudiffu/sage_kernels.py:
// the D pre-pass _sage_attn_d_prepass (:321-349), dK/dV
// _sage_attn_bwd_dkdv_int8 (:805-916) and its tile-masked form (:1491-1615),
// dQ _sage_attn_bwd_dq_int8 (:918-1030) and its tile-masked form (:1617-1722),
// the fp8-QK kernels (:356-590); launchers sage_attention.py:344-458, :534-648.
//
// Operands.  P is recomputed from the forward's per-token codes exactly as the
// forward scores them, s = acc * qd * kd (qd carrying sm_scale*log2(e)),
// p = 2^(s - lse) with the forward's base-2 LSE.  The quantization launch, in
// its backward form, supplies the Q and smoothed-K codes and scales, the rows
// K~ = bf16(k - mean), -D = -rowsum(dO * O) and the LSE padded to whole blocks.
// Q, dO, V and K~ are read as the plain bf16 rows they are.
//
// Rows in LDS.  One copy of a 32-row block serves both as the row operand of
// v_mfma_f32_32x32x16_bf16 (contraction over channels: lane (h, r) reads the
// 16 bytes of row r, channels [16c2 + 8h, +8)) and, through the transposing
// LDS read (ds_read_b64_tr_b16: a group of 16 lanes reads 4 rows x 16 channels
// and each lane gets one channel's 4 rows), as the operand of a contraction
// over rows, in exactly the row order in which a lane of a 32x32 accumulator
// holds its rows (8J + 4h + i): P and dS go from the accumulator registers
// into the next product without a shuffle.  The order of the copy (struct
// Rows) keeps both reads free of bank conflicts and every address one
// lane-constant base plus an immediate.
//
// Two independent workgroups of 4 waves share a CU (at most 80 KB of LDS and
// 256 registers each): they meet at no common barrier, so one's vector work
// (exp, rounding) runs beside the other's matrix work.  Stages pass through a
// two-stage LDS ring filled by direct global -> LDS loads issued one stage
// ahead, one barrier per stage.  Against one 8-wave workgroup per CU whose
// waves all ran the same phase between two barriers, with separate row and
// transposed images of each operand, the kernel takes 1056 -> 862 us at
// 1x30x4416x128 and 1808 -> 1127 us on the packed 1x30x6912 batch with document
// ids, and the preparation that wrote those
// images (51 us) is gone.  What bounds it now is the power limit:
// 27.4 M MFMAs of random data run at 18.2 ns each per SIMD alone (1.79 GHz,
// 489 us), 20.4 ns beside six vector instructions each (546 us).
// Work items are dealt to XCDs in contiguous ranges.  One launch (bwd_kernel)
// runs the dK/dV items, then the dQ items.
//
// dQ pass: a workgroup is the forward's 128-query tile, 32 queries per wave;
// keys stream in steps of 32.  Per wave and step, in the S^T layout (lane
// (h, r) = query r, keys 8J + 4h + i):
//   S^T = K . Q^T (int8 / fp8 MFMA, the forward's operands),
//   dP^T - D = V . dO^T - D (bf16 MFMA started from -D; the wave's dO rows in registers),
//   dS^T = P^T (dP^T - D), dQ += dS . K~ (A = dS from the registers, B = K~ transposed);
// dQ * sm_scale is rounded to bf16 at the end (sage_kernels.py:1720).
// dK/dV pass: a workgroup owns 128 keys, 32 per wave; queries stream in steps
// of 32.  Per wave and step, in the S layout (lane (h, r) = key r, queries
// 8J + 4h + i):
//   S = Q . K^T and dP - D = dO . V^T - D (the wave's K codes and V rows in
//   registers),
//   dS = P (dP - D), dV^T += dO^T . bf16(P), dK^T += Q^T . bf16(dS);
// dK * sm_scale is rounded to bf16 at the end (the reference scales dS before
// its bf16 rounding, :1595: the same relative rounding of the same value).
//
// Both passes skip (query tile, key tile) pairs the reference tile mask turns
// off; with document ids they skip pairs whose summaries show no visible pair,
// and only pairs whose summaries are mixed test every element.  The steps'
// activity is read 64 steps at a time (a lane per step, ballots), so a skipped
// step costs nothing.
#include <type_traits>

#include "sage_common.h"
#include "sage_launch.h"

namespace sage {

namespace {

// 16-byte unit as a native vector: its copies are plain loads and stores.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

template <int QK>
struct BAcc {
  using type = f32x16;
};
template <>
struct BAcc<kQK_INT8> {
  using type = i32x16;
};

// One 32x32 score block from code fragments: rows from `a` (A operand), columns
// from `b`, contracting the D channels (chunks of 32).
template <int D, int QK>
__device__ __forceinline__ typename BAcc<QK>::type score_block(const i32x4* a, const i32x4* b) {
  constexpr int NC = D / 32;
  if constexpr (QK == kQK_INT8) {
    i32x16 acc = i32x16{0};
#pragma unroll
    for (int c = 0; c < NC; ++c) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[c], b[c], acc, 0, 0, 0);
    return acc;
  } else {
    f32x16 acc = f32x16{0};
#pragma unroll
    for (int c = 0; c < NC; c += 2) {
      const i32x8 aa = {a[c][0], a[c][1], a[c][2], a[c][3], a[c + 1][0], a[c + 1][1], a[c + 1][2], a[c + 1][3]};
      const i32x8 bb = {b[c][0], b[c][1], b[c][2], b[c][3], b[c + 1][0], b[c + 1][1], b[c + 1][2], b[c + 1][3]};
      acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(aa, bb, acc, 0, 0, 0, 0, 0, 0);
    }
    return acc;
  }
}

__device__ __forceinline__ bool doc_visible(int dq, int dk) { return dk >= 0 && (dq == dk || dq < 0); }

// Waves of a backward workgroup; two workgroups share a CU.
constexpr int kBwdWaves = 4;
constexpr int kBwdThreads = 64 * kBwdWaves;

// bf16 rows of D channels in LDS: 1 KiB blocks of RPB rows, `stride` bytes
// apart, each one direct global -> LDS load of a wave (64 chunks of 16 bytes)
// that reads 1 KiB of consecutive rows.  Inside a block the rows' 64-byte
// runs are ordered (run, row): four lanes of the load read one run, which
// costs the vector cache a quarter of the accesses that single chunks of four
// rows do (measured: 3.2e8 -> 1.4e8 accesses per launch).  The 16 bytes
// between blocks put rows t and t + RPB in neighbouring chunk columns; with 8
// rows a block (D = 64) rows 4..7 also swap their runs' halves: the 16 lanes
// of a row read and the 32 of a transposed read then touch 256 different
// bytes modulo the banks.
template <int D>
struct Rows {
  static constexpr int RPB = 512 / D;
  static constexpr int stride = 1024 + 16;
  static constexpr int blocks32 = 32 / RPB;
  static constexpr int bytes32 = blocks32 * stride;  // a 32-row block

  static __device__ __forceinline__ int swap(int row_in_block) { return (row_in_block >> 2) * 2; }
  // byte offset in its source block (rows `row_bytes` apart) of the chunk that
  // lane `lane` of the load moves
  static __device__ __forceinline__ int src_off(int lane, int row_bytes) {
    const int t = (lane >> 2) % RPB, run = (lane >> 2) / RPB;
    return t * row_bytes + run * 64 + ((lane & 3) ^ swap(t)) * 16;
  }
  // row operand: lane (h, r) reads row r, channels [16 c2 + 8h, +8) at
  // row_off(lane, c2 % 2) + row_imm(c2)
  static __device__ __forceinline__ int row_off(int lane, int odd) {
    const int h = lane >> 5, r = lane & 31, t = r % RPB;
    return (r / RPB) * stride + t * 64 + ((2 * odd + h) ^ swap(t)) * 16;
  }
  static constexpr int row_imm(int c2) { return c2 / 2 * RPB * 64; }
  // transposed operand: lane (hh, r) gets channel 32c + r of rows 16tt + 8jj +
  // 4hh + 0..3; lane l of a group of 16 reads channels 4 (l % 4) .. +3 (of the
  // group's 16) of row l / 4
  static __device__ __forceinline__ int tr_off(int lane) {
    const int l = lane & 15, g = (lane >> 4) & 1, hh = lane >> 5, t = 4 * hh % RPB + (l >> 2);
    return (4 * hh / RPB) * stride + t * 64 + ((2 * g + ((l & 3) >> 1)) ^ swap(t)) * 16 + (l & 1) * 8;
  }
  static constexpr int tr_imm(int c, int tt, int jj) { return (16 * tt + 8 * jj) / RPB * stride + c * RPB * 64; }
};

// One direct global -> LDS load of 64 chunks: lane l's 16 bytes land at lds + 16 l.
__device__ __forceinline__ void dma_16(uint8_t* lds, __amdgpu_buffer_rsrc_t rs, int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, lds, 16, off, 0, 0, 0);
}

// Rows [0, 32) of `rows` (row_bytes apart; rows past `left` read as zeros)
// into the LDS block at `lds`, by waves `wave`, wave + WAVES, ...  Each load has
// a resource over its own rows, so the lane offset (src_off) is the same for all.
template <int D, int WAVES>
__device__ __forceinline__ void dma_rows32(uint8_t* lds, int wave, int src_off, const uint16_t* rows, int row_bytes,
                                           int64_t left) {
  using R = Rows<D>;
  const int valid = (int)(left > 32 ? 32 : left);
#pragma unroll
  for (int j0 = 0; j0 < R::blocks32; j0 += WAVES) {
    const int j = j0 + wave;
    if (R::blocks32 % WAVES == 0 || j < R::blocks32) {
      const int v = min(valid - j * R::RPB, R::RPB);  // rows of this block
      const __amdgpu_buffer_rsrc_t rs = raw_rsrc(reinterpret_cast<const uint8_t*>(rows) + (int64_t)j * R::RPB * row_bytes,
                                                 v > 0 ? (uint32_t)((v - 1) * row_bytes + 2 * D) : 0u);
      dma_16(lds + j * R::stride, rs, src_off);
    }
  }
}

// 32 consecutive 4-byte values into LDS by one wave: 16-byte aligned ones by
// its first 8 lanes, others (rows past `left` read as zeros) by 32 lanes.
__device__ __forceinline__ void dma_words32(uint8_t* lds, int lane, const void* src) {
  const __amdgpu_buffer_rsrc_t rs = raw_rsrc(src, 128);
  if (lane < 8) dma_16(lds, rs, lane * 16);
}
__device__ __forceinline__ void dma_words32_unaligned(uint8_t* lds, int lane, const void* src, int64_t left) {
  const int valid = (int)(left < 0 ? 0 : left > 32 ? 32 : left);
  const __amdgpu_buffer_rsrc_t rs = raw_rsrc(src, (uint32_t)(valid * 4));
  if (lane < 32) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, lds, 4, lane * 4, 0, 0, 0);
}

// The operand of v_mfma_f32_32x32x16_bf16 that contracts 16 rows (tt): two
// transposed reads of 4 rows each per lane.  `base` is restrict so that the
// reads carry alias information, like plain LDS loads (type-based there):
// without any, the compiler waits for every direct global -> LDS load in
// flight, the next stage's, before each of them.
template <int D>
__device__ __forceinline__ bf16x8 tr_frag(const uint8_t* __restrict__ base, int c, int tt) {
  typedef __attribute__((address_space(3))) s16x4* LdsPtr;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsPtr)(base + Rows<D>::tr_imm(c, tt, 0)));
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsPtr)(base + Rows<D>::tr_imm(c, tt, 1)));
  return __builtin_bit_cast(bf16x8, s16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]});
}

// The first row of dO of head bh (rows dout_rs elements apart).
__device__ __forceinline__ const uint16_t* dout_head(const BwdParams& p, int bh) {
  const int b = bh / p.h;
  return p.dout + b * p.dout_bs + (bh - b * p.h) * p.dout_hs;
}

// Activity of up to 64 steps: bit i of each mask is step base + i.
struct StepMasks {
  uint64_t wg;    // some wave of the workgroup has work
  uint64_t on;    // this wave has work
  uint64_t mixed; // this wave tests every element
};

}  // namespace

// Item of workgroup b of a 1D grid of `total` items: the hardware hands
// workgroup b to XCD b % 8, and each XCD has its own L2, so every XCD takes a
// contiguous range of items (head-major order) and its resident workgroups
// share one head's operands.
__device__ __forceinline__ int xcd_item(int b, int total) {
  constexpr int kXcd = 8;
  const int x = b % kXcd, local = b / kXcd, per = total / kXcd, rem = total % kXcd;
  return x * per + min(x, rem) + local;
}

// ---------------------------------------------------------------------------
// dQ
// ---------------------------------------------------------------------------

// LDS stage of one 32-key step: K codes (row fragments, as stored), V rows,
// K~ rows, per-key K scales, per-key document ids.
template <int D>
struct DqStage {
  static constexpr int offV = 32 * D;
  static constexpr int offT = offV + Rows<D>::bytes32;
  static constexpr int offKd = offT + Rows<D>::bytes32;
  static constexpr int offDoc = offKd + 128;
  static constexpr int bytes = offDoc + 128;
};

// dQ of item (bh, 128-query tile), in `smem` (2 * DqStage<D>::bytes), over
// 32-key steps [s_begin, s_end).  With cut >= 0 the item is cut item `cut`
// (an in-kernel merge as the forward's split items): the half's fp32 dQ goes
// to its slot, and the last half to arrive sums both slots (first half +
// second half) and stores dQ.
template <int D, int QK, int MASK>
__device__ __forceinline__ void dq_item(const BwdParams& p, uint8_t* smem, int item, int s_begin, int s_end, int cut,
                                        int half) {
  using St = DqStage<D>;
  using R = Rows<D>;
  using SAcc = typename BAcc<QK>::type;
  constexpr int NC = D / 32, CPR = D / 8;
  static_assert(kRowsPerWG * D * 2 <= 2 * St::bytes, "the output staging must fit in the ring");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar registers
  const int h = lane >> 5, r = lane & 31;
  const int nq = (int)(p.np / kRowsPerWG);
  const int bh = item / nq, qt = item % nq;
  const int bidx = bh / p.h;
  const int64_t n = p.n, np = p.np;
  const int nt = (int)((n + 63) / 64);
  const int64_t q0 = (int64_t)qt * kRowsPerWG + 32 * wave;
  const bool wave_live = q0 < n;
  const int64_t qrow = q0 + r;

  // ---- per-wave query state -----------------------------------------------------
  i32x4 qf[NC];
  {
    const uint8_t* qb = p.qc + ((int64_t)bh * np + q0) * D;
#pragma unroll
    for (int c = 0; c < NC; ++c) qf[c] = *reinterpret_cast<const i32x4*>(qb + (c * 64 + lane) * 16);
  }
  bf16x8 dof[2 * NC];  // dO[qrow][16c2 + 8h, +8)
  {
    const uint16_t* dr = dout_head(p, bh) + min(qrow, n - 1) * p.dout_rs + 8 * h;
#pragma unroll
    for (int c2 = 0; c2 < 2 * NC; ++c2) dof[c2] = *reinterpret_cast<const bf16x8*>(dr + 16 * c2);
  }
  const float qd = p.qs[(int64_t)bh * np + qrow];
  const float lse_b = p.lse_pad[(int64_t)bh * np + qrow];
  f32x16 nd;  // -D of the lane's query, the start of the dP sums
  {
    const float d = p.neg_delta[(int64_t)bh * np + qrow];
#pragma unroll
    for (int e = 0; e < 16; ++e) nd[e] = d;
  }
  const int dq_doc = (MASK & 2) ? (qrow < n ? p.doc[(int64_t)bidx * n + qrow] : -1) : 0;
  f32x16 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = f32x16{0};

  // ---- active steps: tile t = s / 2 against the workgroup's 128 queries and this wave's 32 ----
  int4 qsum128 = make_int4(0, 0, 0, 0), qsum32 = make_int4(0, 0, 0, 0);
  if constexpr (MASK & 2) {
    qsum128 = load_uniform(p.q_sum128, (int64_t)bidx * nq + qt);
    qsum32 = load_uniform(p.q_sum, (int64_t)bidx * (np / 32) + (q0 >> 5));
  }
  StepMasks sm{0, 0, 0};
  int sm_base = -1;
  auto find = [&](int s) __attribute__((always_inline)) -> int {
    if constexpr (MASK == 0) return s;
    while (s < s_end) {
      if ((s & ~63) != sm_base) {
        sm_base = s & ~63;
        const int t = (sm_base + lane) >> 1;
        bool wg = sm_base + lane < s_end, on = wg, mixed = false;
        if constexpr (MASK & 1)
          wg = wg && p.tile_mask[(int64_t)bh * p.mask_stride_z + (int64_t)qt * p.mask_nkv + min(t, nt - 1)] != 0;
        on = wg;
        if constexpr (MASK & 2) {
          const int4 ks = p.kv_sum[(int64_t)bidx * nt + min(t, nt - 1)];
          const int c = classify(qsum32, ks);
          on = wg && c != 0;
          mixed = c == 2;
          wg = wg && classify(qsum128, ks) != 0;
        }
        sm.wg = __ballot(wg);
        sm.on = __ballot(on);
        sm.mixed = __ballot(mixed);
      }
      const uint64_t m = sm.wg >> (s & 63);
      if (m) return s + __builtin_ctzll(m);
      s = sm_base + 64;
    }
    return s_end;
  };

  // ---- staging -------------------------------------------------------------------
  const int src_off = R::src_off(lane, 2 * D);
  auto load_step = [&](int s, int stage) __attribute__((always_inline)) {
    const int64_t key0 = (int64_t)s * 32;
    uint8_t* sb = smem + stage * St::bytes;
    dma_chunks_buf<2 * D, kBwdWaves>(sb, wave, lane, raw_rsrc(p.kc + ((int64_t)bh * np + key0) * D, 32 * D), 0);
    dma_rows32<D, kBwdWaves>(sb + St::offV, wave, src_off, p.v + ((int64_t)bh * n + key0) * D, 2 * D, n - key0);
    dma_rows32<D, kBwdWaves>(sb + St::offT, wave, src_off, p.kt + ((int64_t)bh * n + key0) * D, 2 * D, n - key0);
    if (wave == 2) dma_words32(sb + St::offKd, lane, p.ks + (int64_t)bh * np + key0);
    if constexpr (MASK & 2) {
      if (wave == 3) dma_words32_unaligned(sb + St::offDoc, lane, p.doc + (int64_t)bidx * n + key0, n - key0);
    }
  };
  const int row_off[2] = {R::row_off(lane, 0), R::row_off(lane, 1)}, tr_off = R::tr_off(lane);

  int s = find(s_begin);
  if (s < s_end) load_step(s, 0);
  int stage = 0;
  while (s < s_end) {
    const bool on = wave_live && (MASK == 0 || ((sm.on >> (s & 63)) & 1));
    const bool mixed = (MASK & 2) && ((sm.mixed >> (s & 63)) & 1);
    const int sn = find(s + 1);
    wait_vmem();
    __syncthreads();  // stage complete; every wave is past the step that used the other stage
    if (sn < s_end) load_step(sn, stage ^ 1);
    if (on) {
      const uint8_t* sb = smem + stage * St::bytes;
      // S^T = K . Q^T for keys (lane-local rows) x this wave's queries
      i32x4 ka[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) ka[c] = reinterpret_cast<const i32x4*>(sb)[c * 64 + lane];
      const SAcc sc = score_block<D, QK>(ka, qf);
      // dP^T - D = V . dO^T - D, its MFMAs issued under the exponentials of P
      f32x16 dp = nd;
      const f32x4* kdl = reinterpret_cast<const f32x4*>(sb + St::offKd);
      const int4* dkl = reinterpret_cast<const int4*>(sb + St::offDoc);
      const int kmax = (int)min((int64_t)32, n - (int64_t)s * 32);  // valid keys of this step
      const uint8_t* vl = sb + St::offV;
      bf16x8 vf[2 * NC];
      vf[0] = *reinterpret_cast<const bf16x8*>(vl + row_off[0]);
      vf[1] = *reinterpret_cast<const bf16x8*>(vl + row_off[1]);
      f32x4 kd4[4];
#pragma unroll
      for (int J = 0; J < 4; ++J) kd4[J] = kdl[2 * J + h];
      float pr[16];
      // s - lse = acc * (qd * kd) - lse
      constexpr int kPer = 16 / (2 * NC);  // scores per MFMA
#pragma unroll
      for (int c2 = 0; c2 < 2 * NC; ++c2) {
        __builtin_amdgcn_sched_barrier(0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[c2], dof[c2], dp, 0, 0, 0);
        if (c2 + 2 < 2 * NC) vf[c2 + 2] = *reinterpret_cast<const bf16x8*>(vl + row_off[c2 & 1] + R::row_imm(c2 + 2));
#pragma unroll
        for (int e = kPer * c2; e < kPer * c2 + kPer; ++e)
          pr[e] = __builtin_amdgcn_exp2f(fmaf((float)sc[e], qd * kd4[e >> 2][e & 3], -lse_b));
      }
      __builtin_amdgcn_sched_barrier(0);
      // keys past N (the last step only) and, in mixed pairs, hidden keys: p = 0
      if (kmax < 32 || mixed) {
#pragma unroll
        for (int J = 0; J < 4; ++J) {
          int4 dk4 = make_int4(0, 0, 0, 0);
          if constexpr (MASK & 2) dk4 = dkl[2 * J + h];
          const int dk[4] = {dk4.x, dk4.y, dk4.z, dk4.w};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            bool vis = 8 * J + 4 * h + i < kmax;
            if constexpr (MASK & 2) vis = vis && doc_visible(dq_doc, dk[i]);
            pr[4 * J + i] = vis ? pr[4 * J + i] : 0.0f;
          }
        }
      }
      // dQ += dS . K~ (A = dS, rounded to bf16), the first 16 keys' products under the others' rounding
      const uint8_t* tl = sb + St::offT + tr_off;
      bf16x8 dsa[2];
#pragma unroll
      for (int e = 0; e < 8; ++e) dsa[0][e] = (__bf16)(pr[e] * dp[e]);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dsa[0], tr_frag<D>(tl, c, 0), acc[c], 0, 0, 0);
#pragma unroll
        for (int e = 8 / NC * c; e < 8 / NC * (c + 1); ++e) dsa[1][e] = (__bf16)(pr[8 + e] * dp[8 + e]);
      }
#pragma unroll
      for (int c = 0; c < NC; ++c)
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dsa[1], tr_frag<D>(tl, c, 1), acc[c], 0, 0, 0);
    }
    stage ^= 1;
    s = sn;
  }
  wait_vmem();
  __syncthreads();  // the ring is free

  // ---- epilogue: dQ * sm_scale -> bf16 ------------------------------------------------
  // acc lane (h, r) holds channel 32c + r of rows 8J + 4h + i (element 4J + i)
  if (cut >= 0) {
    // a half of a cut item: its dQ through to the coherence point, complete
    // before it counts; the last half sums the two slots in key order
    constexpr int kSlot = 4 * NC * 16 * 64;
    uint32_t* slots = reinterpret_cast<uint32_t*>(p.dq_part + (int64_t)cut * 2 * kSlot);
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        __hip_atomic_store(slots + half * kSlot + ((wave * NC + c) * 16 + e) * 64 + lane, __float_as_uint(acc[c][e]),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    wait_vmem();
    __syncthreads();
    int* last = reinterpret_cast<int*>(smem);
    if (tid == 0) *last = arrive_last(p.dq_ctr + cut, p.dq_tag, 2) ? 1 : 0;
    __syncthreads();
    if (*last == 0) return;
    auto ld = [](const uint32_t* a) __attribute__((always_inline)) {
      return __uint_as_float(__hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    };
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int at = ((wave * NC + c) * 16 + e) * 64 + lane;
        acc[c][e] = ld(slots + at) + ld(slots + kSlot + at);
      }
    if (tid == 0)
      __hip_atomic_store(p.dq_ctr + cut, p.dq_tag << 8, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();  // every wave has read `last` before the staging below reuses the LDS
  }
  uint16_t* stg = reinterpret_cast<uint16_t*>(smem) + wave * 32 * D;  // the wave's own rows
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int row = 8 * (e >> 2) + 4 * h + (e & 3);
      stg[row * D + 32 * c + r] = f32_to_bf16_rne(acc[c][e] * p.sm_scale);
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 32 * CPR / 64; ++i) {
    const int x = lane + 64 * i, row = x / CPR, ch = x % CPR;
    const int64_t q = q0 + row;
    if (q < n)
      *reinterpret_cast<uint4*>(p.dq + ((int64_t)bh * n + q) * D + ch * 8) =
          reinterpret_cast<const uint4*>(stg)[x];
  }
}

// ---------------------------------------------------------------------------
// dK, dV
// ---------------------------------------------------------------------------

// LDS stage of one 32-query step: Q codes (row fragments), Q rows, dO rows,
// per-query Q scale, LSE, -D, document ids.
template <int D>
struct DkvStage {
  static constexpr int offQ = 32 * D;
  static constexpr int offDo = offQ + Rows<D>::bytes32;
  static constexpr int offQd = offDo + Rows<D>::bytes32;
  static constexpr int offLse = offQd + 128;
  static constexpr int offNd = offLse + 128;
  static constexpr int offDoc = offNd + 128;
  static constexpr int bytes = offDoc + 128;
};

// The wave's 32 V rows, the column operand of dP in every step, stay in
// registers (D/4 of them), except with document ids at D = 128: the mixed
// steps' registers leave no room there (4-8 spilled), so the rows stay in LDS
// behind the ring.  Measured at 1x30x4416x128 without ids: 903.8 -> 891.4 us.
template <int D, int MASK>
constexpr bool kVInRegs = D == 64 || (MASK & 2) == 0;

// LDS of a dK/dV item: two step stages, then the V rows if they are there.
template <int D, int MASK>
constexpr int kDkvLds = 2 * DkvStage<D>::bytes + (kVInRegs<D, MASK> ? 0 : kBwdWaves * Rows<D>::bytes32);

// dK, dV of item (bh, 128-key block), in `smem` (kDkvLds<D, MASK>).  Wave w owns
// keys 32w .. +31 of the block.
template <int D, int QK, int MASK>
__device__ __forceinline__ void dkdv_item(const BwdParams& p, uint8_t* smem, int item) {
  using St = DkvStage<D>;
  using R = Rows<D>;
  using SAcc = typename BAcc<QK>::type;
  constexpr int NC = D / 32, CPR = D / 8;
  constexpr int kOutStride = 2 * D + 16;  // bytes of a staged output row: no bank is hit by two rows' 8-byte pieces
  static_assert(kBwdWaves * 32 * kOutStride <= 2 * St::bytes, "the output staging must fit in the ring");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar registers
  const int h = lane >> 5, r = lane & 31;
  const int nkb = (int)(p.np / kRowsPerWG);
  const int bh = item / nkb, kb = item % nkb;
  const int bidx = bh / p.h;
  const int64_t n = p.n, np = p.np;
  const int nkv = (int)((n + 63) / 64);
  const int nsteps = (int)((n + 31) / 32);  // 32-query steps holding a query below N
  const int64_t k0 = (int64_t)kb * kRowsPerWG + 32 * wave;
  const int64_t krow = k0 + r;
  const bool wave_live = k0 < n;

  // ---- per-wave key state -------------------------------------------------------------
  i32x4 kf[NC];
  {
    const uint8_t* kbp = p.kc + ((int64_t)bh * np + k0) * D;
#pragma unroll
    for (int c = 0; c < NC; ++c) kf[c] = *reinterpret_cast<const i32x4*>(kbp + (c * 64 + lane) * 16);
  }
  const int src_off = R::src_off(lane, 2 * D), do_off = R::src_off(lane, (int)(2 * p.dout_rs));
  const int tr_off = R::tr_off(lane);
  const uint16_t* dout = dout_head(p, bh);
  const int row_off[2] = {R::row_off(lane, 0), R::row_off(lane, 1)};
  bf16x8 vf[2 * NC];                                         // V[krow][16c2 + 8h, +8)
  uint8_t* vlds = smem + 2 * St::bytes + wave * R::bytes32;  // or the wave's V rows
  if constexpr (kVInRegs<D, MASK>) {
    const uint16_t* vr = p.v + ((int64_t)bh * n + min(krow, n - 1)) * D + 8 * h;
#pragma unroll
    for (int c2 = 0; c2 < 2 * NC; ++c2) vf[c2] = *reinterpret_cast<const bf16x8*>(vr + 16 * c2);
  } else if (wave_live) {
    dma_rows32<D, 1>(vlds, 0, src_off, p.v + ((int64_t)bh * n + k0) * D, 2 * D, n - k0);
  }
  const float kd = p.ks[(int64_t)bh * np + krow];
  const int dk_doc = (MASK & 2) ? (krow < n ? p.doc[(int64_t)bidx * n + krow] : -1) : 0;
  f32x16 dva[NC], dka[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    dva[c] = f32x16{0};
    dka[c] = f32x16{0};
  }

  // ---- active steps: 32-query block s against the workgroup's two key tiles, this wave's one ----
  int4 ksum[2] = {make_int4(0, 0, 0, 0), make_int4(0, 0, 0, 0)};
  if constexpr (MASK & 2) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      ksum[i] = 2 * kb + i < nkv ? load_uniform(p.kv_sum, (int64_t)bidx * nkv + 2 * kb + i)
                                 : make_int4(0x7fffffff, -0x7fffffff, 0, 0);
  }
  StepMasks sm{0, 0, 0};
  int sm_base = -1;
  auto find = [&](int s) __attribute__((always_inline)) -> int {
    if constexpr (MASK == 0) return s;
    while (s < nsteps) {
      if ((s & ~63) != sm_base) {
        sm_base = s & ~63;
        const int st = min(sm_base + lane, nsteps - 1);
        bool on0 = sm_base + lane < nsteps, on1 = on0 && 2 * kb + 1 < nkv;
        if constexpr (MASK & 1) {
          const uint8_t* m = p.tile_mask + (int64_t)bh * p.mask_stride_z + (int64_t)(st >> 2) * p.mask_nkv + 2 * kb;
          on0 = on0 && m[0] != 0;
          on1 = on1 && m[on1 ? 1 : 0] != 0;
        }
        bool mixed = false;
        if constexpr (MASK & 2) {
          const int4 qs = p.q_sum[(int64_t)bidx * (np / 32) + st];
          const int c0 = classify(qs, ksum[0]), c1 = classify(qs, ksum[1]);
          on0 = on0 && c0 != 0;
          on1 = on1 && c1 != 0;
          mixed = (wave >> 1 ? c1 : c0) == 2;
        }
        sm.wg = __ballot(on0 || on1);
        sm.on = __ballot(wave >> 1 ? on1 : on0);
        sm.mixed = __ballot(mixed);
      }
      const uint64_t m = sm.wg >> (s & 63);
      if (m) return s + __builtin_ctzll(m);
      s = sm_base + 64;
    }
    return nsteps;
  };

  // ---- staging -----------------------------------------------------------------------
  auto load_step = [&](int s, int stage) __attribute__((always_inline)) {
    const int64_t m0 = (int64_t)s * 32;
    uint8_t* sb = smem + stage * St::bytes;
    dma_chunks_buf<2 * D, kBwdWaves>(sb, wave, lane, raw_rsrc(p.qc + ((int64_t)bh * np + m0) * D, 32 * D), 0);
    dma_rows32<D, kBwdWaves>(sb + St::offDo, wave, do_off, dout + m0 * p.dout_rs, (int)(2 * p.dout_rs), n - m0);
    dma_rows32<D, kBwdWaves>(sb + St::offQ, wave, src_off, p.q + ((int64_t)bh * n + m0) * D, 2 * D, n - m0);
    if (wave < 3) {
      const float* src = wave == 0 ? p.qs : wave == 1 ? p.lse_pad : p.neg_delta;
      dma_words32(sb + St::offQd + wave * 128, lane, src + (int64_t)bh * np + m0);
    } else if constexpr (MASK & 2) {
      dma_words32_unaligned(sb + St::offDoc, lane, p.doc + (int64_t)bidx * n + m0, n - m0);
    }
  };

  int s = find(0);
  if (s < nsteps) load_step(s, 0);
  int stage = 0;
  while (s < nsteps) {
    const bool on = wave_live && (MASK == 0 || ((sm.on >> (s & 63)) & 1));
    const bool mixed = (MASK & 2) && ((sm.mixed >> (s & 63)) & 1);
    const int sn = find(s + 1);
    wait_vmem();
    __syncthreads();  // stage complete; every wave is past the step that used the other stage
    if (sn < nsteps) load_step(sn, stage ^ 1);
    if (on) {
      const uint8_t* sb = smem + stage * St::bytes;
      const f32x4* qdl = reinterpret_cast<const f32x4*>(sb + St::offQd);
      const f32x4* lsl = reinterpret_cast<const f32x4*>(sb + St::offLse);
      const f32x4* ndl = reinterpret_cast<const f32x4*>(sb + St::offNd);
      const int4* dql = reinterpret_cast<const int4*>(sb + St::offDoc);
      // S = Q . K^T: rows = queries, columns = this wave's keys
      i32x4 qa[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) qa[c] = reinterpret_cast<const i32x4*>(sb)[c * 64 + lane];
      const SAcc sacc = score_block<D, QK>(qa, kf);
      // dP - D = dO . V^T - D
      f32x16 dp;
#pragma unroll
      for (int J = 0; J < 4; ++J) {
        const f32x4 d4 = ndl[2 * J + h];
#pragma unroll
        for (int i = 0; i < 4; ++i) dp[4 * J + i] = d4[i];
      }
      // ... its MFMAs issued under the exponentials of P
      const uint8_t* dol = sb + St::offDo;
      bf16x8 wf[2 * NC];
      auto dpfrag = [&](int c2) __attribute__((always_inline)) {
        wf[c2] = *reinterpret_cast<const bf16x8*>(dol + row_off[c2 & 1] + R::row_imm(c2));
        if constexpr (!kVInRegs<D, MASK>)
          vf[c2] = *reinterpret_cast<const bf16x8*>(vlds + row_off[c2 & 1] + R::row_imm(c2));
      };
      dpfrag(0);
      dpfrag(1);
      float pr[16];
      bf16x8 pb[2], db[2];
      // s - lse = acc * (qd * kd) - lse; keys past N need no test: their
      // column only feeds their own dK / dV rows, which are not stored
      constexpr int kPer = 16 / (2 * NC);  // scores per MFMA
      f32x4 qd4, ls4;
#pragma unroll
      for (int c2 = 0; c2 < 2 * NC; ++c2) {
        __builtin_amdgcn_sched_barrier(0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[c2], vf[c2], dp, 0, 0, 0);
        if (c2 + 2 < 2 * NC) dpfrag(c2 + 2);
#pragma unroll
        for (int e = kPer * c2; e < kPer * c2 + kPer; ++e) {
          const int J = e >> 2, i = e & 3;
          if (i == 0) {
            qd4 = qdl[2 * J + h];
            ls4 = lsl[2 * J + h];
          }
          pr[e] = __builtin_amdgcn_exp2f(fmaf((float)sacc[e], qd4[i] * kd, -ls4[i]));
          if constexpr ((MASK & 2) == 0) pb[e >> 3][e & 7] = (__bf16)pr[e];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (MASK & 2) {
        if (mixed) {  // hidden keys: p = 0
#pragma unroll
          for (int J = 0; J < 4; ++J) {
            const int4 dq4 = dql[2 * J + h];
            const int dqd[4] = {dq4.x, dq4.y, dq4.z, dq4.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) pr[4 * J + i] = doc_visible(dqd[i], dk_doc) ? pr[4 * J + i] : 0.0f;
          }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) pb[e >> 3][e & 7] = (__bf16)pr[e];
      }
      // dV^T += dO^T . P under the rounding of dS, then dK^T += Q^T . dS
      const uint8_t* tdl = sb + St::offDo + tr_off;
      const uint8_t* tql = sb + St::offQ + tr_off;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          dva[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag<D>(tdl, c, tt), pb[tt], dva[c], 0, 0, 0);
#pragma unroll
          for (int e = 8 / NC * c; e < 8 / NC * (c + 1); ++e) db[tt][e] = (__bf16)(pr[8 * tt + e] * dp[8 * tt + e]);
        }
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int c = 0; c < NC; ++c)
          dka[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag<D>(tql, c, tt), db[tt], dka[c], 0, 0, 0);
    }
    stage ^= 1;
    s = sn;
  }
  wait_vmem();
  __syncthreads();  // the ring is free

  // ---- epilogue: lane (h, r) holds key r, channels 32c + 8J + 4h + i; rows staged in LDS ----
  uint8_t* stg = smem + wave * 32 * kOutStride;  // the wave's own rows
  auto store_rows = [&](const f32x16* x, float scale, uint16_t* out) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int J = 0; J < 4; ++J) {
        uint2 w;
        w.x = f32_to_bf16_rne(x[c][4 * J + 0] * scale) | ((uint32_t)f32_to_bf16_rne(x[c][4 * J + 1] * scale) << 16);
        w.y = f32_to_bf16_rne(x[c][4 * J + 2] * scale) | ((uint32_t)f32_to_bf16_rne(x[c][4 * J + 3] * scale) << 16);
        *reinterpret_cast<uint2*>(stg + r * kOutStride + (32 * c + 8 * J + 4 * h) * 2) = w;
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 32 * CPR / 64; ++i) {
      const int y = lane + 64 * i, row = y / CPR, ch = y % CPR;
      if (k0 + row < n)
        *reinterpret_cast<uint4*>(out + ((int64_t)bh * n + k0 + row) * D + ch * 8) =
            *reinterpret_cast<const uint4*>(stg + row * kOutStride + ch * 16);
    }
    __syncthreads();
  };
  store_rows(dva, 1.0f, p.dv);
  store_rows(dka, p.sm_scale, p.dk);
}

// The two gradient passes in one launch: workgroups [0, kv_wgs) take the
// dK/dV items (kv_wgs = items rounded up to a multiple of 8, the extra ones
// exit), the next `items` the dQ items, of which the last p.dq_split take the
// first key-tile half of their item, and the dq_split after those the second
// halves (dispatched last, the short pieces fill the launch's end).  The passes are independent, so the
// dQ items fill the CUs the last dK/dV round leaves idle, and the shorter
// items come last.  Each part deals its items to the XCDs like a launch of
// its own (xcd_item): kv_wgs is a multiple of the XCD count, so a dQ
// workgroup's XCD is its index within the part modulo 8.
template <int D, int MASK>
constexpr int kBwdLds = kDkvLds<D, MASK> > 2 * DqStage<D>::bytes ? kDkvLds<D, MASK> : 2 * DqStage<D>::bytes;
static_assert(2 * kBwdLds<128, 2> <= 160 * 1024, "two workgroups per CU");

template <int D, int QK, int MASK>
__global__ void __launch_bounds__(kBwdThreads, 2) bwd_kernel(BwdParams p, int items, int kv_wgs) {
  __shared__ __attribute__((aligned(16))) uint8_t smem[kBwdLds<D, MASK>];
  const int wg = (int)blockIdx.x;
  if (wg < kv_wgs) {
    if (wg < items) dkdv_item<D, QK, MASK>(p, smem, xcd_item(wg, items));
    return;
  }
  const int steps = (int)((p.n + 31) / 32), mid = (int)((p.n + 63) / 64) / 2 * 2;  // 32-key steps; whole tiles first
  const int j = wg - kv_wgs, whole = items - p.dq_split;
  const bool second = j >= items, cut = j >= whole;
  dq_item<D, QK, MASK>(p, smem, xcd_item(second ? j - p.dq_split : j, items), second ? mid : 0,
                       cut && !second ? mid : steps, cut ? (second ? j - items : j - whole) : -1, second ? 1 : 0);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

template <int D, int QK, int MASK>
hipError_t launch_bwd_t(const BwdParams& p, int64_t bh, hipStream_t st) {
  const int64_t items = p.np / kRowsPerWG * bh;  // per pass, in xcd_item order
  const int64_t kv_wgs = (items + 7) / 8 * 8;
  hipLaunchKernelGGL((bwd_kernel<D, QK, MASK>), dim3((unsigned)(kv_wgs + items + p.dq_split)), dim3(kBwdThreads), 0,
                     st, p, (int)items, (int)kv_wgs);
  return hipGetLastError();
}

template <int D>
hipError_t launch_bwd_d(int qk, int mask, const BwdParams& p, int64_t bh, hipStream_t st) {
#define SAGE_B_CASE(QK_, M_) \
  if (qk == QK_ && mask == M_) return launch_bwd_t<D, QK_, M_>(p, bh, st);
  SAGE_B_CASE(0, 0) SAGE_B_CASE(0, 1) SAGE_B_CASE(0, 2) SAGE_B_CASE(0, 3)
  SAGE_B_CASE(1, 0) SAGE_B_CASE(1, 1) SAGE_B_CASE(1, 2) SAGE_B_CASE(1, 3)
#undef SAGE_B_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_bwd(int qk, int mask, const BwdParams& p, int64_t d, int64_t bh, hipStream_t st) {
  if (d == 128) return launch_bwd_d<128>(qk, mask, p, bh, st);
  if (d == 64) return launch_bwd_d<64>(qk, mask, p, bh, st);
  return hipErrorInvalidValue;
}

}  // namespace sage
