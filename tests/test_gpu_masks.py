"""GPU: the device mask builders against the oracle (bit-exact), and the
packed plumbing end to end: a mask built on the device drives the attention
exactly like the host-built one, and exact document ids make a packed batch
equal to running each image alone."""

import math
import random

import pytest
import torch

from oracle import sage_oracle as O

pytestmark = pytest.mark.gpu


def _segments(rng, n_min=200):
    segs = [rng.choice([rng.randint(1, 700), 32 * rng.randint(1, 40), 64 * rng.randint(1, 20)])
            for _ in range(rng.randint(1, 5))]
    while sum(segs) < n_min:
        segs.append(rng.randint(1, 300))
    return segs


@pytest.mark.parametrize("seed", range(4))
def test_device_tile_mask_matches_oracle(cuda, seed):
    from futudiffu_amd import block_mask as BM
    rng = random.Random(100 + seed)
    rows, want = [], []
    for _ in range(3):
        segs = _segments(rng)
        total = sum(segs) + rng.choice([0, rng.randint(1, 200)])
        rows.append((segs, total))
    n = max(t for _, t in rows)
    docs = []
    for segs, total in rows:
        doc = O.packed_document_ids(segs, total) + [-1] * (n - total)
        docs.append(doc)
        want.append(O.tile_mask_from_doc(doc, pad_fill=0))
    print(f"tile mask seed={seed} n={n}", flush=True)
    d = torch.tensor(docs, dtype=torch.int32, device=cuda)
    got = BM.build_block_mask_device(d)
    one = BM.build_block_mask_device(d[0].contiguous())
    fill = BM.build_block_mask_device(d, pad_fill=7)
    torch.cuda.synchronize()
    assert torch.equal(got.cpu(), torch.stack(want))
    assert torch.equal(one.cpu(), want[0])
    assert torch.equal(fill.cpu(), torch.stack([O.tile_mask_from_doc(x, pad_fill=7) for x in docs]))


@pytest.mark.parametrize("seed", range(4))
def test_device_doc_ids_from_cu_seqlens_match_oracle(cuda, seed):
    from futudiffu_amd import block_mask as BM
    rng = random.Random(200 + seed)
    nseg = rng.randint(1, 7)
    cus = []
    for _ in range(2):
        cu = [rng.choice([0, 0, rng.randint(1, 40)])]
        for _ in range(nseg):
            cu.append(cu[-1] + rng.choice([0, rng.randint(1, 500)]))
        cus.append(cu)
    n = max(c[-1] for c in cus) + rng.randint(0, 90)
    print(f"cu_seqlens seed={seed} n={n} segments={nseg}", flush=True)
    got = BM.doc_ids_from_cu_seqlens(torch.tensor(cus, dtype=torch.int32, device=cuda), n)
    one = BM.doc_ids_from_cu_seqlens(torch.tensor(cus[0], dtype=torch.int32, device=cuda), n)
    torch.cuda.synchronize()
    assert got.cpu().tolist() == [O.doc_ids_from_cu_seqlens(c, n) for c in cus]
    assert one.cpu().tolist() == [O.doc_ids_from_cu_seqlens(cus[0], n)]


def test_packing_info_device_mask_drives_attention_like_host_mask(cuda):
    """A padded packed plan (two images in 4288 tokens): the mask built on the
    device from document_id equals the host-built reference mask, so the
    attention outputs are bit-identical."""
    from types import SimpleNamespace

    from futudiffu_amd import block_mask as BM
    from futudiffu_amd import sage_attention as SA
    segs = [(0, 96, 96, 1184), (1280, 64, 1344, 1152)]
    lens = [96 + 1184, 64 + 1152]
    doc = torch.tensor(O.packed_document_ids(lens, 4288), dtype=torch.int32, device=cuda)
    info = SimpleNamespace(segments=segs, total_len=4288, document_id=doc)
    dev_mask = BM.build_block_mask_from_packing_info(info, device=cuda)
    host_mask = BM.build_block_mask(lens, 4288, device="cpu")
    assert torch.equal(dev_mask.cpu(), host_mask)
    B, H, N, D = 1, 2, 4288, 128
    q, k, v = (t.to(cuda) for t in O.make_inputs(B, H, N, D, seed=71))
    a, la = SA.sage_attn_forward_masked_with_lse(q, k, v, dev_mask, 1.0 / math.sqrt(D))
    b, lb = SA.sage_attn_forward_masked_with_lse(q, k, v, host_mask.to(cuda), 1.0 / math.sqrt(D))
    torch.cuda.synchronize()
    assert torch.equal(a.view(torch.int16), b.view(torch.int16)) and torch.equal(la, lb)


@pytest.mark.parametrize("qk,pv", [("int8", "fp8"), ("fp8", "bf16"), ("int8", "bf16"), ("fp8", "fp8")])
def test_packed_exact_ids_equal_serial_images(cuda, qk, pv):
    """Three images of 64-aligned lengths packed into one sequence (plus 64
    padding tokens), masked by exact ids from device cu_seqlens.  Without K
    smoothing every code depends only on its own token (V scales on its own
    64-token block), and each image's rows see exactly its own key tiles in
    the same order, so the packed rows equal each image run alone, bit for
    bit, outputs and LSE."""
    from futudiffu_amd import block_mask as BM
    from futudiffu_amd import sage_attention as SA
    lens = [640, 1216, 1152]
    n = sum(lens) + 64
    B, H, D = 1, 2, 128
    q, k, v = (t.to(cuda) for t in O.make_inputs(B, H, n, D, seed=73))
    cu = torch.tensor([0, 640, 1856, 3008], dtype=torch.int32, device=cuda)
    doc = BM.doc_ids_from_cu_seqlens(cu, n)
    print(f"packed vs serial {qk}/{pv} lens={lens}", flush=True)
    out, lse = SA.sage_forward(q, k, v, qk=qk, pv=pv, smooth_k=False, doc_ids=doc)
    off = 0
    for s in lens:
        sl = slice(off, off + s)
        o1, l1 = SA.sage_forward(q[:, :, sl].contiguous(), k[:, :, sl].contiguous(), v[:, :, sl].contiguous(),
                                 qk=qk, pv=pv, smooth_k=False)
        torch.cuda.synchronize()
        got = out[:, :, sl].contiguous()
        bad = got.view(torch.int16) != o1.view(torch.int16)
        assert not bad.any(), (f"segment at {off}: {int(bad.sum())} outputs differ, "
                               f"max {(got.float() - o1.float()).abs().max().item():.3g}")
        assert torch.equal(lse.view(B * H, n)[:, sl].cpu(), l1.cpu()), f"segment at {off}: LSE differs"
        off += s


@pytest.mark.parametrize("qk,pv", [("int8", "fp8"), ("int8", "bf16"), ("fp8", "fp8")])
def test_packed_tile_mask_equal_serial_images(cuda, qk, pv):
    """Three images of 128-aligned lengths packed into one sequence, masked by
    the reference tile mask built on the device from their document ids; for
    aligned images that mask is exactly block diagonal.  Without K smoothing
    each image's rows see exactly their own key tiles, in the order of the
    image run alone, so outputs and LSE equal the serial runs bit for bit.
    The tile-mask loop starts its int8 score chains from zero like the
    unmasked one; the exact-id test above pins the document-id loop, which
    starts them from c0, to the same scores."""
    from futudiffu_amd import block_mask as BM
    from futudiffu_amd import sage_attention as SA
    lens = [640, 1152, 1280]
    n = sum(lens)
    B, H, D = 1, 2, 128
    q, k, v = (t.to(cuda) for t in O.make_inputs(B, H, n, D, seed=79))
    doc = torch.tensor(O.packed_document_ids(lens, n), dtype=torch.int32, device=cuda)
    mask = BM.build_block_mask_device(doc)
    print(f"packed tile mask vs serial {qk}/{pv} lens={lens}", flush=True)
    out, lse = SA.sage_forward(q, k, v, qk=qk, pv=pv, smooth_k=False, block_mask=mask)
    off = 0
    for s in lens:
        sl = slice(off, off + s)
        o1, l1 = SA.sage_forward(q[:, :, sl].contiguous(), k[:, :, sl].contiguous(), v[:, :, sl].contiguous(),
                                 qk=qk, pv=pv, smooth_k=False)
        torch.cuda.synchronize()
        got = out[:, :, sl].contiguous()
        bad = got.view(torch.int16) != o1.view(torch.int16)
        assert not bad.any(), (f"segment at {off}: {int(bad.sum())} outputs differ, "
                               f"max {(got.float() - o1.float()).abs().max().item():.3g}")
        assert torch.equal(lse.view(B * H, n)[:, sl].cpu(), l1.cpu()), f"segment at {off}: LSE differs"
        off += s


@pytest.mark.parametrize("pv,D", [("bf16", 128), ("fp8", 128), ("bf16", 64)])
def test_tile_masked_tail_split(cuda, pv, D):
    """65 heads of 1000 tokens are 520 items: with room in the workspace the
    last 8 run as up to four shares of their active tiles each.  A 3D mask
    gives the split items 0 to 16 active tiles, scattered ones among them; the
    results agree with the unsplit launch (a workspace of the masked size) to
    the rounding of P in another frame, rows without a key give 0 and -inf,
    and two heads match the oracle."""
    from futudiffu_amd import _lib
    from futudiffu_amd import sage_attention as SA
    B, H, N = 1, 65, 1000
    nq, nkv = 8, 16
    lib = _lib.load()
    q, k, v = O.make_inputs(B, H, N, D, seed=91)
    g = torch.Generator().manual_seed(92)
    mask = (torch.rand(H, nq, nkv, generator=g) < 0.5).to(torch.uint8)
    for i, count in enumerate([0, 1, 3, 4, 7, 8, 15, 16]):  # the last head's items are the split ones
        mask[H - 1, i] = 0
        mask[H - 1, i, torch.randperm(nkv, generator=g)[:count]] = 1
    print(f"masked tail split int8/{pv} D={D}", flush=True)
    qz = SA.quantize_qkv(q.to(cuda), k.to(cuda), v.to(cuda), qk="int8", pv=pv)
    mg = mask.to(cuda)
    out, lse = SA.attn_from_quantized(qz, B, H, block_mask=mg)
    out2, lse2 = SA.attn_from_quantized(qz, B, H, block_mask=mg)
    wsb = int(lib.sage_attn_masked_workspace_bytes(B, H, N, D))
    assert wsb < int(lib.sage_attn_workspace_bytes(B, H, N, D))
    ws = torch.empty(wsb, dtype=torch.uint8, device=cuda)
    o1 = torch.empty_like(out)
    l1 = torch.empty_like(lse)
    _lib.check(lib.sage_attn_fwd(
        qz.q_codes.data_ptr(), qz.q_scale.data_ptr(), qz.k_codes.data_ptr(), qz.k_scale.data_ptr(),
        qz.v_op.data_ptr(), SA._ptr(qz.v_scale), B, H, N, D, 0, SA._PV[pv], 0, mg.data_ptr(), nq * nkv, nq, nkv, None,
        ws.data_ptr(), wsb, o1.data_ptr(), 0, l1.data_ptr(), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(out, out2) and torch.equal(lse, lse2)
    assert torch.equal(out[:, :H - 1], o1[:, :H - 1]) and torch.equal(lse[:H - 1], l1[:H - 1])
    assert not out[0, H - 1, :128].float().any() and torch.isinf(lse[H - 1, :128]).all()
    assert (out.float() - o1.float()).abs().max().item() <= 8e-3
    fin = torch.isfinite(l1)
    assert torch.equal(fin, torch.isfinite(lse)) and (lse[fin] - l1[fin]).abs().max().item() <= 1e-4
    for hh in (0, H - 1):
        sl = slice(hh, hh + 1)
        live = mask[hh].sum(1) > 0
        m1 = mask[hh:hh + 1].clone()
        m1[0, ~live] = 1
        want, wl, _ = O.sage_forward(q[:, sl], k[:, sl], v[:, sl], 1.0 / math.sqrt(D), "int8", pv, "token", True, m1)
        see = live.repeat_interleave(128)[:N]
        got = out[:, sl].float().cpu()[:, :, see]
        assert (got - want.float()[:, :, see]).abs().max().item() <= 2e-2
        assert O.cosine(got, want[:, :, see]) >= 0.999
        assert (lse[hh].cpu()[see] - wl[0][see]).abs().max().item() <= 2e-3


def test_tile_masked_few_items_cut(cuda):
    """Two heads of 1921 tokens are 32 items of 31 key tiles, cut into up to
    three shares of at least 12 active tiles: a 3D mask gives the items 0 to 31
    active tiles, scattered ones, on both sides of 24.  Against the uncut launch
    (a workspace of the masked size), to the rounding of P in another frame."""
    from futudiffu_amd import _lib
    from futudiffu_amd import sage_attention as SA
    B, H, N, D, nq, nkv = 1, 2, 1921, 128, 16, 31
    lib = _lib.load()
    q, k, v = (t.to(cuda) for t in O.make_inputs(B, H, N, D, seed=95))
    g = torch.Generator().manual_seed(96)
    mask = torch.zeros(H, nq, nkv, dtype=torch.uint8)
    for i in range(H * nq):
        mask[i // nq, i % nq, torch.randperm(nkv, generator=g)[:i]] = 1
    mask[0, 0] = 1
    mask[1, 3] = 0
    mg = mask.to(cuda)
    live = mask.sum(2).repeat_interleave(128, 1)[:, :N] > 0
    for pv in ("bf16", "fp8"):
        print(f"masked few items int8/{pv}", flush=True)
        qz = SA.quantize_qkv(q, k, v, qk="int8", pv=pv)
        out, lse = SA.attn_from_quantized(qz, B, H, block_mask=mg)
        wsb = int(lib.sage_attn_masked_workspace_bytes(B, H, N, D))
        assert wsb < int(lib.sage_attn_workspace_bytes(B, H, N, D))
        ws = torch.empty(wsb, dtype=torch.uint8, device=cuda)
        o1, l1 = torch.empty_like(out), torch.empty_like(lse)
        _lib.check(lib.sage_attn_fwd(
            qz.q_codes.data_ptr(), qz.q_scale.data_ptr(), qz.k_codes.data_ptr(), qz.k_scale.data_ptr(),
            qz.v_op.data_ptr(), SA._ptr(qz.v_scale), B, H, N, D, 0, SA._PV[pv], 0, mg.data_ptr(), nq * nkv, nq, nkv,
            None, ws.data_ptr(), wsb, o1.data_ptr(), 0, l1.data_ptr(), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert torch.equal(torch.isfinite(lse).cpu(), live) and torch.equal(torch.isfinite(l1).cpu(), live)
        assert not out[0][~live.to(cuda)].float().any()
        # the bound of test_tile_masked_tail_split: one bf16 step of an output up to 2
        assert (out.float() - o1.float()).abs().max().item() <= 8e-3
        fin = live.to(cuda)
        assert (lse[fin] - l1[fin]).abs().max().item() <= 1e-4


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("lens", [[64, 64], [40, 88], [40, 150], [100, 220], [130, 258], [70, 1, 400]])
def test_bf16_document_ids_on_the_pipelined_loop(cuda, lens, D):
    """bf16 P.V with document ids: the tiles some wave does not see whole go
    through the general loop, the rest (here none to six, a ragged last one)
    through the pipelined one; padding keys put mixed tiles before whole ones in
    the second sample."""
    from futudiffu_amd import sage_attention as SA
    n = sum(lens)
    doc = torch.cat([torch.full((s,), i, dtype=torch.int32) for i, s in enumerate(lens)])
    pad = torch.zeros(n, dtype=torch.int32)
    pad[lens[0] // 2: lens[0]] = -1
    ids = torch.stack([doc, pad])
    B, H = 2, 2
    q, k, v = O.make_inputs(B, H, n, D, seed=300 + n)
    print(f"bf16 document ids {lens} D={D}", flush=True)
    out, lse = SA.sage_forward(q.to(cuda), k.to(cuda), v.to(cuda), qk="int8", pv="bf16", doc_ids=ids.to(cuda))
    torch.cuda.synchronize()
    want, wl, _ = O.sage_forward(q, k, v, None, "int8", "bf16", "token", True, None, ids)
    # the output bounds of every variant against the reference scheme
    assert (out.cpu().float() - want.float()).abs().max().item() <= 2e-2
    assert O.cosine(out.cpu(), want) >= 0.999
    assert (lse.cpu() - wl.view_as(lse.cpu())).abs().max().item() <= 2e-3


@pytest.mark.parametrize("H,D,pv,lens", [(24, 128, "fp8", [500, 1000]), (52, 128, "bf16", [1600]),
                                         (60, 64, "bf16", [1537]), (60, 128, "fp8", [1500, 37])])
def test_tile_masked_launches_cut(cuda, H, D, pv, lens):
    """Launches whose items are cut: 32 past one per CU, of 16 active tiles, 164
    past a round in two shares each, and 268 of which 85 are cut.  Against the uncut launch (a workspace of the masked size), to the
    rounding of P in another frame."""
    from futudiffu_amd import _lib
    from futudiffu_amd import sage_attention as SA
    B, N = 1, sum(lens)
    lib = _lib.load()
    q, k, v = (t.to(cuda) for t in O.make_inputs(B, H, N, D, seed=N + D))
    mg = O.build_block_mask(lens, N).to(cuda)
    print(f"masked launch cut {B}x{H}x{N}x{D} {pv}", flush=True)
    qz = SA.quantize_qkv(q, k, v, qk="int8", pv=pv)
    out, lse = SA.attn_from_quantized(qz, B, H, block_mask=mg)
    wsb = int(lib.sage_attn_masked_workspace_bytes(B, H, N, D))
    ws = torch.empty(wsb, dtype=torch.uint8, device=cuda)
    o1, l1 = torch.empty_like(out), torch.empty_like(lse)
    _lib.check(lib.sage_attn_fwd(
        qz.q_codes.data_ptr(), qz.q_scale.data_ptr(), qz.k_codes.data_ptr(), qz.k_scale.data_ptr(),
        qz.v_op.data_ptr(), SA._ptr(qz.v_scale), B, H, N, D, 0, SA._PV[pv], 0, mg.data_ptr(), 0, mg.shape[0],
        mg.shape[1], None, ws.data_ptr(), wsb, o1.data_ptr(), 0, l1.data_ptr(),
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert not torch.equal(out, o1)  # some item is cut
    # the bound of test_tile_masked_tail_split: one bf16 step of an output up to 2
    assert (out.float() - o1.float()).abs().max().item() <= 8e-3
    assert (lse - l1).abs().max().item() <= 1e-4


@pytest.mark.parametrize("B,H,D,lens", [(1, 30, 128, [1003, 771, 1297]), (1, 30, 128, [500, 400, 600]),
                                        (2, 30, 64, [1337]), (4, 30, 128, [300])])
def test_tile_masked_launches_left_whole(cuda, B, H, D, lens):
    """Launches whose items are not cut, with room for partials: 208 items past a
    round of at most 21 active tiles (two shares take 24), items of at most 10
    below one round (they are cut from 12 on), 148 items past a round of 21
    tiles, items of 5 tiles.  The bits of the launch that has no room."""
    from futudiffu_amd import _lib
    from futudiffu_amd import sage_attention as SA
    N = sum(lens)
    lib = _lib.load()
    q, k, v = (t.to(cuda) for t in O.make_inputs(B, H, N, D, seed=N))
    mg = O.build_block_mask(lens, N).to(cuda)
    print(f"masked launch left whole {B}x{H}x{N}x{D}", flush=True)
    qz = SA.quantize_qkv(q, k, v, qk="int8", pv="bf16")
    out, lse = SA.attn_from_quantized(qz, B, H, block_mask=mg)
    wsb = int(lib.sage_attn_masked_workspace_bytes(B, H, N, D))
    ws = torch.empty(wsb, dtype=torch.uint8, device=cuda)
    o1, l1 = torch.empty_like(out), torch.empty_like(lse)
    _lib.check(lib.sage_attn_fwd(
        qz.q_codes.data_ptr(), qz.q_scale.data_ptr(), qz.k_codes.data_ptr(), qz.k_scale.data_ptr(),
        qz.v_op.data_ptr(), None, B, H, N, D, 0, 0, 0, mg.data_ptr(), 0, mg.shape[0], mg.shape[1], None,
        ws.data_ptr(), wsb, o1.data_ptr(), 0, l1.data_ptr(), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(out, o1) and torch.equal(lse, l1)
