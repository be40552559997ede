// Host-side launcher declarations shared by the kernel files and the C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace sage {

struct AttnParams {
  const uint8_t* qc;
  const float* qs;
  const uint8_t* kc;
  const float* ks;
  const uint8_t* vin;
  const float* vs;
  const uint8_t* tile_mask;
  int64_t mask_stride_z;
  int64_t mask_nkv;
  const int32_t* doc;
  const int4* kv_sum;  // [B][nT]   (min doc, max doc, #valid, #padding) over keys < N
  const int4* q_sum;     // [B][Np/32] same over queries < N
  const int4* q_sum128;  // [B][Np/128] same over queries < N
  // [B][Np/128] with document ids, per 128-row query tile: (first scheduled
  // key tile, one past the last scheduled key tile that some live wave of
  // the tile does not see whole (0 if none), one past the last scheduled key
  // tile, 0); an item with no scheduled tile has first = nT, last = 0
  const int4* doc_range;
  // with document ids: [0].x the number of listed split query tiles, [1 + e].x
  // = b * nq + qt of entry e < heavy_max (doc_prefix_kernel); the first
  // heavy_max * h workgroups take them
  int4* heavy;
  int heavy_max;
  uint16_t* out;
  // element strides of out per batch, head and row: [B,H,N,D] is
  // (H*N*D, N*D, D), [B,N,H,D] is (N*H*D, D, H*D)
  int64_t out_bs, out_hs, out_rs;
  float* lse;
  int64_t n;
  int64_t np;
  int h;           // heads per batch
  int bh;          // B * H
  int nt;          // key tiles: ceil(N / 64)
  int light_last;  // last 128-row query tile holds <= 64 rows: schedule those items last
  // without document ids: the items past n_whole (in schedule order) are cut
  // into (with a tile mask, at most) split_parts key-tile ranges, merged by the
  // last range to finish or, unmasked, by a second kernel
  int n_whole;
  int split_parts;
  float* part;  // (items - n_whole) * split_parts slots of kPartFloats<D> floats
  // in-kernel merge: one arrival counter per split item (the last piece to
  // arrive merges the item); null: merge_split_kernel merges after the launch.
  // A counter holds merge_tag << 8 | pieces arrived; the merging piece resets
  // it to merge_tag << 8, so a graph replay with the same tag counts from 0.
  uint64_t* merge_ctr;
  uint64_t merge_tag;
  // parity only (int8 QK, unmasked): int32 [BH, Np, Np] receives the S^T
  // accumulators of every tile the kernel's own loop consumes (row = query)
  int32_t* s_dump;
  // tile mask alone: a split item is cut into at most (active tiles) /
  // share_min pieces, and not at all below share_from active tiles
  int share_from;
  int share_min;
};

// Split query tiles (document ids) that the first workgroups of a launch take
// (AttnParams::heavy): kHeavyMax * h workgroups are reserved for them.
constexpr int kHeavyMax = 2;

// Resident workgroups of the attention kernel on MI355X: 256 CUs x 2 (three a CU
// with bf16 P.V at D = 64, which the splits below do not count on).
constexpr int kResidentWGs = 512;

// Floats of one partial slot: O of 128 rows x D (fp32, lane order), then the
// per-lane reference point and row-sum halves of the 4 waves.
template <int D>
constexpr int64_t kPartFloats = 128 * D + 2 * 256;

// Split of an unmasked launch of n_items 128-row items of nt key tiles:
// whole items fill complete rounds of the resident workgroups; the items of
// the last, partial round are cut into `parts` ranges of key tiles (at most
// 4), chosen to minimize (rounds the pieces take) x (tiles per piece + 2
// tiles of pipeline start).  The cap of 4 is measured: at 1050 items of 69
// tiles, 4 pieces beat 8 (257.6 vs 260.0 us) and 2 (271.7 us), since the
// partials' traffic and merge grow with the piece count and the pieces run
// beside the second round's last items.
//
// Launches of less than one round: an item alone on a CU runs about 1.4x
// faster than one of two sharing it (its waves have the SIMDs' issue slots to
// themselves), so when up to 128 items spill past one per CU, the first 256
// stay whole and the spilled items are cut into key-tile pieces that share
// the CUs with them: 4 pieces (at least 2 tiles each) while every piece still
// fits the one round of resident workgroups, else as many as fit, at least 2.
// Measured at 20 tiles with a separate merge kernel: 2 pieces, 260 items
// 43.5 -> 34.8 us, 300 items 41.6 -> 36.9, 350 items 41.5 -> 39.1; 400 items
// lose, 42.1 -> 55.7.  With the merge inside the attention kernel, 300 items:
// 34.4 us in 2 pieces, 31.7 / 31.6 in 3 / 4, 33.1 in 5; cutting every item
// costs more than it balances (in 2 / 3 / 4 pieces, by this rule last: 300 items
// of 20 tiles 51.2 / 51.0 / 62.0 against 30.8 us, 288 of 64 tiles 99.3 / 90.5 /
// 98.6 against 75.5, 390 of 26 tiles, all whole, 64.8 / 72.5 / 89.4 against 47.6).
//
// Launches of no more items than CUs: each item walks all its tiles alone (1.05
// us a tile) while CUs idle, so every item is cut, from 24 tiles on.  At most
// 128 items: pieces of 10 tiles or more, as many as there are CUs for (3x3000,
// 72 items of 47 tiles: 53.6 us whole, 30.6 in 3 pieces, 36.8 / 38.7 in 4 / 6
// that share CUs), since a piece's start, partial and share of the merge cost
// some 7 us (16x1024, 16 tiles: 21.3 -> 23.5 in 2; 2x2048, 32 tiles: 37.4 ->
// 24.0 in 3 of 10, 27.4 in 2 of 16, 26.3 in 5 of 6).  More items: the pieces
// must share CUs, which pays from 48 tiles (D=64: 140 items of 69 tiles 61.5 ->
// 42.4 us, 240 of 60 tiles 54.3 -> 50.2, 192 of 32 tiles 30.6 -> 31.6).  The
// partials stay within the allocation-free entry point's scratch (small_slots),
// so that it takes every such launch: at D=128 up to 123 items.
struct TailSplit {
  int64_t whole;
  int parts;
};

// Partial slots (128 x D + 512 floats) in 16 MiB less 64 KiB for the rest of
// the workspace, whose summaries take under 32 KiB at 256 items.
inline constexpr int64_t small_slots(int64_t d) { return ((16 << 20) - (64 << 10)) / ((128 * d + 512) * 4); }

inline TailSplit tail_split(int64_t n_items, int64_t nt, int64_t d) {
  TailSplit t{n_items, 1};
  constexpr int64_t kCUs = kResidentWGs / 2;
  if (n_items <= 0) return t;  // a workspace size asked for an empty batch
  if (n_items <= kCUs) {
    const bool share = n_items > kCUs / 2;
    if (nt < (share ? 48 : 24)) return t;
    const int64_t room = share ? (int64_t)kResidentWGs : kCUs, slots = small_slots(d);
    int64_t parts = (room < slots ? room : slots) / n_items;
    parts = parts < 8 ? parts : 8;
    parts = parts < nt / 10 ? parts : nt / 10;
    return parts > 1 ? TailSplit{0, (int)parts} : t;
  }
  if (n_items > kCUs && n_items < kResidentWGs) {
    const int64_t spill = n_items - kCUs;
    if (spill <= 128 && nt >= 2) {
      int64_t parts = kCUs / spill;  // pieces that fit the round
      parts = parts < 4 ? parts : 4;
      parts = parts < nt / 2 ? parts : nt / 2;
      t = TailSplit{kCUs, (int)(parts > 2 ? parts : 2)};
    }
    return t;
  }
  const int64_t rest = n_items >= kResidentWGs ? n_items % kResidentWGs : 0;
  if (rest == 0) return t;
  int64_t best = (rest + kResidentWGs - 1) / kResidentWGs * (nt + 2);
  const int pmax = (int)(nt < 4 ? nt : 4);
  for (int p = 2; p <= pmax; ++p) {
    const int64_t cost = (rest * p + kResidentWGs - 1) / kResidentWGs * ((nt + p - 1) / p + 2);
    if (cost < best) {
      best = cost;
      t.parts = p;
    }
  }
  if (t.parts > 1) t.whole = n_items - rest;
  return t;
}

// The split of a tile-masked launch without document ids: tail_split's items
// (reduced to `split` by attn_workspace's limit), each cut into equal shares of
// its active tiles by the kernel, which alone knows the mask.
//
// Beside full rounds, or past one item per CU, a share takes at least 4 tiles,
// and items of fewer than 12 stay whole: a piece's start, partial and share of
// the merge cost more than so short an item leaves idle.  Where every item is
// cut, or more than 128 beside full rounds (whose pieces share CUs), it takes at
// least 12.  A launch whose items cannot have two shares is not split
// (4x30x300x128, 5 tiles: 13.2 us whole, 14.8 with workgroups that only exit).
// Measured over 356 launches of 1 to 4 documents of 800 to 6912 tokens together,
// geometric mean of the attention kernel's time over the uncut launch's, for bf16
// and fp8 P.V (slower ones by 12 % at most):
//   past one per CU       D=128 0.94, 0.89;  D=64 0.90, 0.87
//   1 to 128 past a round D=128 0.97, 0.95;  D=64 0.94, 0.93
//   more                  D=128 0.98, 0.96;  D=64 0.98, 0.96
// Shares of 4 everywhere are 3 to 9 % slower than these where more are past a
// round, and 1 to 2 % elsewhere (short items).
struct MaskedSplit {
  TailSplit split;
  int share_from, share_min;
};

// Bytes of workspace a tile-masked split may take, of the unmasked launch's:
// two pieces of 256 items at D = 128.  The allocation-free entry point's array
// has them, so that every entry with the room cuts the same items.
inline constexpr size_t kMaskedSplitBytes = (size_t)34 << 20;

inline MaskedSplit masked_split(TailSplit split, int64_t n_items, int64_t nt) {
  const bool few = split.whole != 0 && n_items % kResidentWGs - (n_items < kResidentWGs ? split.whole : 0) <= 128;
  MaskedSplit m{split, few ? 12 : 0, few ? 4 : 12};
  if (m.split.parts > nt / m.share_min) m.split.parts = (int)(nt / m.share_min);
  if (m.split.parts < 2) m.split = TailSplit{n_items, 1};
  return m;
}

// Inputs of the q/k/v producer (QKV split + per-head RMSNorm + Flux RoPE +
// transpose, fused_kernels.py:271-390).  With qkv set, the quantization reads
// the projection output and applies the producer itself; with qkv null it
// reads bf16 q, k, v [BH, N, D].
// Heads per slab unit of the producer kernels (one pass of tokens for this
// many heads of a batch in one workgroup).
constexpr int kSlabHeads = 8;

struct ProdArgs {
  const uint16_t* qkv;  // bf16 [B, N, 3*H*D]
  const float* qw;      // RMSNorm weights of q and k, fp32 [D]
  const float* kw;
  const float* freqs;   // fp32 [B*N, D/2, 2, 2]: [[cos, -sin], [sin, cos]] per channel pair
  int h;
  int bh;               // B*H
  float eps;
};

hipError_t launch_quantize(int qk, int pv, int gran, bool smooth, const uint16_t* q, const uint16_t* k,
                           const uint16_t* v, int64_t bh, int64_t n, int64_t d, float fold, double* ws,
                           uint8_t* qc, float* qs, uint8_t* kc, float* ks, uint8_t* vout, float* vs,
                           uint16_t* kmean, const ProdArgs& prod, hipStream_t st);
// The quantization in its backward form: per-token codes and scales of Q and K
// and the K mean, and the backward's own operands: the rows kt = bf16(k - mean)
// [BH, N, D] (with smoothing), neg_delta = -rowsum(dout * out) and the LSE with
// +inf for rows without gradient, both [BH, Np].
struct BwdPrep {
  uint16_t* kt;
  const uint16_t* dout;
  int64_t dout_bs, dout_hs, dout_rs;  // element strides per batch, head and row
  const uint16_t* out;
  int64_t out_bs, out_hs, out_rs;
  const float* lse;
  float* neg_delta;
  float* lse_pad;
  int h;  // heads per batch
};
hipError_t launch_quantize_bwd(int qk, bool smooth, const uint16_t* q, const uint16_t* k, int64_t bh, int64_t n,
                               int64_t d, float fold, double* ws, uint8_t* qc, float* qs, uint8_t* kc, float* ks,
                               uint16_t* kmean, const BwdPrep& prep, hipStream_t st);
hipError_t launch_qkv_postprocess(const ProdArgs& prod, int64_t bh, int64_t n, int64_t d, uint16_t* q_out,
                                  uint16_t* k_out, uint16_t* v_out, hipStream_t st);
// Gradient of the producer with respect to its input (fused_kernels.py:711-783):
// gq, gk, gv bf16 [BH, N, D] -> dqkv bf16 [B, N, 3*H*D].
hipError_t launch_qkv_postprocess_bwd(const ProdArgs& prod, int64_t bh, int64_t n, int64_t d, const uint16_t* gq,
                                      const uint16_t* gk, const uint16_t* gv, uint16_t* dqkv, hipStream_t st);
size_t quant_workspace_bytes(int64_t bh, int64_t n, int64_t d);
int64_t quant_grid_units(int64_t bh, int64_t n, int64_t d, int64_t h_producer);

hipError_t launch_attn(int qk, int pv, int gran, int mask, const AttnParams& p, int64_t d, int nb, hipStream_t st);
// Per-batch document-id summaries (min doc, max doc, #valid, #padding) of every
// 64-key tile ([nb][ceil(n/64)]), 32-row block ([nb][Np/32]) and 128-row block
// ([nb][Np/128]).
// The scheduled key-tile range of each 128-row query tile and one past the
// last key tile that some live wave of it does not see whole (the doc_range
// entries), from the summaries (after launch_doc_summaries).
// Also lists the query tiles whose live waves see different key-tile ranges
// (heavy, when not null; see AttnParams::heavy).
hipError_t launch_doc_prefix(const int4* kv_sum, const int4* q_sum, const int4* q_sum128, int64_t n, int nb,
                             int4* range, int4* heavy, hipStream_t st);
// heavy (may be null): the split-query-tile list to empty before launch_doc_prefix.
hipError_t launch_doc_summaries(const int32_t* doc, int64_t n, int nb, int4* kv_sum, int4* q_sum, int4* q_sum128,
                                int4* heavy, hipStream_t st);
// Workspace of one attention call: the doc-id summaries, then the partial
// slots of the tail split.
struct AttnWorkspace {
  size_t doc_off, heavy_off, part_off, ctr_off, bytes;
  TailSplit split;
};
// `masked`: a launch that splits no item (document ids, or a tile mask in a
// workspace without room for partials).  `limit` (0: none): the partials
// kept within it, by fewer pieces an item up to one item per CU and by fewer
// items beyond (then no more pieces than CUs); none if that leaves under two
// pieces.
AttnWorkspace attn_workspace(int64_t b, int64_t h, int64_t n, int64_t d, bool masked = false, size_t limit = 0);
size_t attn_workspace_bytes(int64_t b, int64_t h, int64_t n, int64_t d, bool masked = false);
hipError_t launch_tile_mask(const int32_t* doc, int64_t nb, int64_t n, int32_t pad_fill, uint8_t* mask,
                            hipStream_t st);

// Backward (sage_kernels.py:321-349, :805-1030, :1491-1722).  Codes and
// scales are the quantization's per-token outputs ([BH, Np] layout, Q scale
// with sm_scale*log2(e)); q, v, kt (K~, the smoothed K: k itself without
// smoothing) and the gradients are plain rows [BH, N, D], dout rows of D at the
// given strides; lse_pad and neg_delta are [BH, Np] (launch_quantize_bwd).
struct BwdParams {
  const uint8_t* qc;
  const float* qs;
  const uint8_t* kc;
  const float* ks;
  const uint16_t* q;
  const uint16_t* kt;
  const uint16_t* v;
  const uint16_t* dout;
  int64_t dout_bs, dout_hs, dout_rs;  // element strides per batch, head and row (AttnParams::out_bs)
  const float* lse_pad;
  const float* neg_delta;
  const uint8_t* tile_mask;
  int64_t mask_stride_z;
  int64_t mask_nkv;
  const int32_t* doc;     // [B, N] document ids (mask bit 2)
  const int4* kv_sum;     // their summaries: [B][ceil(N/64)] key tiles,
  const int4* q_sum;      // [B][Np/32] and [B][Np/128] query blocks
  const int4* q_sum128;
  uint16_t* dq;
  uint16_t* dk;
  uint16_t* dv;
  int64_t n, np;
  int h;
  float sm_scale;
  // the last dq_split dQ items of the launch (a multiple of 8) run as two
  // key-tile halves, dispatched last: fp32 partial dQ slots [dq_split][2]
  // of 128 * D floats, one arrival counter per cut item (dq_tag << 8 | halves
  // arrived; the merging half resets it to dq_tag << 8)
  int dq_split;
  float* dq_part;
  uint64_t* dq_ctr;
  uint64_t dq_tag;
};

// dQ items of a backward launch cut in two key-tile halves (at most; a
// multiple of 8, so both halves of an item run on one XCD).
constexpr int kBwdDqSplit = 64;

hipError_t launch_bwd(int qk, int mask, const BwdParams& p, int64_t d, int64_t bh, hipStream_t st);
hipError_t launch_doc_from_cu(const int32_t* cu, int64_t nb, int64_t nseg, int64_t n, int32_t* doc,
                              hipStream_t st);

}  // namespace sage
