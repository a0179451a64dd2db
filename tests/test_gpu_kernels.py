"""Kernel-level parity of the HIP path against the CPU oracle (GPU only).

Bit-exact: permute gather/scatter, operand preparation, top-k from identical
fp32 scores. Tolerance: pooled tiles (hi+lo split, rel 2e-5), block scores
(rel 2e-3 against fp32), attention output in fp32 (max-abs 2e-2, mean-rel 1e-3
against fp32 masked-dense attention; mean-rel = mean|out - ref| / mean|ref|).
"""
import math

import numpy as np
import pytest
import torch

from dfsattn_amd import ops
from dfsattn_amd.layout import ScoringLayout, hunyuan_policy, wan_policy, dense_policy
from oracle import dfs_oracle as orc

pytestmark = pytest.mark.gpu


def _swap23(s):
    return (s & ~12) | ((s & 4) << 1) | ((s & 8) >> 1)


def vt_reference(v_perm_padded: torch.Tensor, dtype) -> torch.Tensor:
    """[H, R, D] (execution order, zero rows past L) -> [H, R/128, D, 128]
    with tokens of each 16-group in swap23 order."""
    h, r, d = v_perm_padded.shape
    idx = torch.tensor([_swap23(s) for s in range(16)])
    x = v_perm_padded.view(h, r // 128, 8, 16, d)[:, :, :, idx, :]
    return x.reshape(h, r // 128, 128, d).transpose(2, 3).to(dtype).contiguous()


def mean_rel(out, ref):
    return float((out.double() - ref.double()).abs().mean() / ref.double().abs().mean())


@pytest.mark.parametrize("dtype,d,length,n", [
    (torch.bfloat16, 128, 67, 61),   # the reference's own Triton-permute test shape
    (torch.float32, 64, 1000, 1000),
    (torch.float16, 3, 257, 200),    # 6-byte rows: 2-byte vector path
])
def test_permute_gather_scatter_bit_exact(dev, dtype, d, length, n):
    torch.manual_seed(40)
    src = torch.randn((1, 3, length, d), dtype=dtype)
    perm = torch.randperm(n)
    perm_d = perm.to(dev, torch.int32)
    out = ops.permute_gather(src.to(dev), perm_d, rows=n + 5).cpu()
    assert torch.equal(out[:, :, :n], src[:, :, perm])
    assert torch.count_nonzero(out[:, :, n:]) == 0
    # inverse permutation: scatter of the gathered rows restores the source rows
    back = torch.zeros_like(src).to(dev)
    ops.permute_scatter(out[:, :, :n].contiguous().to(dev), perm_d, out=back)
    back = back.cpu()
    assert torch.equal(back[:, :, perm], src[:, :, perm])
    untouched = torch.ones(length, dtype=torch.bool)
    untouched[perm] = False
    assert torch.count_nonzero(back[:, :, untouched]) == 0


@pytest.mark.parametrize("case", ["wan_tail", "wan_even", "hunyuan_text", "hunyuan_no_text", "d64_tile32",
                                  "tile8", "d64_tile64", "q8_k64", "q128_k4_text", "d64_q64_k32", "no_q_operand"])
def test_prepare_qkv_matches_oracle(dev, case):
    heads, d, tile, dtype, pv = 2, 128, 16, torch.bfloat16, torch.float16
    k_tile = None
    q_operand = case != "no_q_operand"
    if case == "wan_tail":
        length, video = 1000, 1000
    elif case == "wan_even":
        length, video = 1024, 1024
    elif case == "hunyuan_text":
        length, video = 1000 + 60, 1000
    elif case == "hunyuan_no_text":
        length, video = 1000, 1000
    elif case == "tile8":  # tile sizes the scorer does not take are still prepared
        length, video, tile = 1000 + 40, 1000, 8
    elif case == "d64_tile64":
        length, video, d, tile = 900, 900, 64, 64
    elif case == "q8_k64":  # unequal query and key tiles (attention_wan.py:94-95)
        length, video, tile, k_tile = 1000, 1000, 8, 64
    elif case == "q128_k4_text":
        length, video, tile, k_tile = 1000 + 60, 1000, 128, 4
    elif case == "d64_q64_k32":
        length, video, d, tile, k_tile = 900, 900, 64, 64, 32
    elif case == "no_q_operand":  # Q only pooled (the attention kernel reads it from the input)
        length, video = 1000 + 60, 1000
    else:
        length, video, d, tile, pv = 777, 777, 64, 32, torch.bfloat16
    torch.manual_seed(7)
    q, k, v = (torch.randn((1, heads, length, d)).to(dtype) for _ in range(3))
    vperm = torch.randperm(video)
    perm, _ = orc.full_permutation(vperm, length)
    layout = ScoringLayout(length, video, tile, k_tile=k_tile)
    prep = ops.prepare_qkv(q.to(dev), k.to(dev), v.to(dev), perm.to(dev, torch.int32), layout, operand_dtype=pv,
                           q_operand=q_operand)
    qp, kp, vp = (orc.apply_permutation(x, perm) for x in (q, k, v))
    R = layout.rows
    pad = lambda x: torch.cat([x[0], x.new_zeros(heads, R - length, d)], dim=1)
    assert prep.k_perm.dtype == pv  # f16 operands: exact bf16 -> f16 rounding
    if q_operand:
        assert prep.q_perm.dtype == pv and torch.equal(prep.q_perm.cpu(), pad(qp).to(pv))
    else:
        assert prep.q_perm is None and prep.q_src is not None
    assert torch.equal(prep.k_perm.cpu(), pad(kp).to(pv))
    assert torch.equal(prep.v_t.cpu(), vt_reference(pad(vp), pv))
    if prep.exps is not None:  # bf16 inputs inside the f16 range: no head is rescaled
        assert int(prep.exps.abs().sum().item()) == 0
    qt, kt = orc.pooled_tiles(qp, kp, tile, 128, video, k_tile=k_tile)
    for hi, lo, ref in ((prep.q_hi, prep.q_lo, qt[0]), (prep.k_hi, prep.k_lo, kt[0])):
        got = hi.cpu().float() + lo.cpu().float()
        assert got.shape == ref.shape
        assert torch.allclose(got, ref, rtol=2e-5, atol=1e-6), float((got - ref).abs().max())


def test_prepare_rescales_heads_beyond_f16(dev):
    """bf16 inputs rounded to f16 operands: a head holding a finite value
    beyond the f16 range is stored as x * 2^-e, e the smallest exponent with
    max|x| * 2^-e < 2^15 (1e6 = 2^19.93 -> e = 5), bit-exactly; every other
    head keeps plain rounding and exponent 0. bf16 operands keep the bits and
    carry no exponents."""
    heads, length, d = 3, 300, 64
    layout = ScoringLayout(length, length, 16)
    ident = torch.arange(length, dtype=torch.int32, device=dev)
    for which in range(3):
        qkv = [torch.randn((1, heads, length, d)).to(torch.bfloat16) for _ in range(3)]
        qkv[which][0, 1, 123, 7] = 1.0e6
        prep = ops.prepare_qkv(*(x.to(dev) for x in qkv), ident, layout, pool=False)
        exps = prep.exps.cpu()
        want = torch.zeros(3, heads, dtype=torch.int32)
        want[which, 1] = 5
        assert torch.equal(exps, want), (which, exps)
        R = layout.rows
        scaled = [x[0].float() for x in qkv]
        scaled[which][1] *= 2.0 ** -5
        for t, got in enumerate((prep.q_perm, prep.k_perm)):
            ref = torch.cat([scaled[t].to(torch.float16), torch.zeros(heads, R - length, d, dtype=torch.float16)], 1)
            assert torch.equal(got.cpu(), ref), (which, t)
        pad = torch.cat([scaled[2], scaled[2].new_zeros(heads, R - length, d)], 1)
        assert torch.equal(prep.v_t.cpu(), vt_reference(pad, torch.float16)), which
        keep = ops.prepare_qkv(*(x.to(dev) for x in qkv), ident, layout, operand_dtype=torch.bfloat16, pool=False)
        assert keep.exps is None
        assert torch.equal(keep.q_perm.cpu()[:, :length], qkv[0][0])


@pytest.mark.parametrize("pv", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize("q_operand", [True, False])
def test_bsa_fwd_keeps_inputs_beyond_f16(dev, pv, q_operand):
    """Heads with q, k or v beyond the f16 range (q * scale * log2(e) beyond
    it too, so rows carry their own power of two) against fp32 masked
    attention of the same bf16 inputs."""
    from dfsattn_amd.workloads import DfsConfig, synth_qkv
    heads, d, length = 4, 128, 1000
    cfg = DfsConfig("big", (1, 1, length), heads, d, torch.bfloat16, seed=31)
    q, k, v = (x.clone() for x in synth_qkv(cfg))
    v[:, 0] = (v[:, 0].float() * 3.0e5).to(torch.bfloat16)        # V beyond f16
    k[:, 1] = (k[:, 1].float() * 2.0e5).to(torch.bfloat16)        # K beyond f16
    q[:, 2] = (q[:, 2].float() * 1.0e6).to(torch.bfloat16)        # Q, and Q * c, beyond f16
    q[:, 3, :500] = (q[:, 3, :500].float() * 4.0e5).to(torch.bfloat16)  # only some rows of a head
    k[:, 3] = (k[:, 3].float() * 1.0e2).to(torch.bfloat16)
    g = torch.Generator().manual_seed(32)
    nb = math.ceil(length / 128)
    mask = torch.rand((heads, nb, nb), generator=g) < 0.5
    mask[:, torch.arange(nb), torch.arange(nb)] = True
    layout = ScoringLayout(length, length, 16)
    ident = torch.arange(length, dtype=torch.int32, device=dev)
    prep = ops.prepare_qkv(q.to(dev), k.to(dev), v.to(dev), ident, layout, operand_dtype=pv, pool=False,
                           q_operand=q_operand)
    row_ptr, col_idx = ops.mask_to_csr(mask.to(dev))
    got = ops.bsa_fwd(prep, row_ptr, col_idx, out_dtype=torch.float32).cpu()
    ref = orc.masked_attention(q, k, v, mask)
    assert bool(torch.isfinite(got).all())
    for h in range(heads):
        rel = mean_rel(got[:, h], ref[:, h])
        print(f"head {h} ({pv}): mean-rel {rel:.2e}", flush=True)
        assert rel <= (1e-3 if pv == torch.float16 else 3e-3), h


def _random_scores(heads, rows, cols, seed, ties=False):
    g = torch.Generator().manual_seed(seed)
    s = torch.rand((heads, rows, cols), generator=g)
    if ties:
        s = torch.round(s * 8) / 8  # many exact ties, some straddling the k-th place
    return s


@pytest.mark.parametrize("cols,ratio,ties", [(591, 0.3, False), (8, 0.3, False), (100, 0.05, True),
                                             (931, 0.3, True), (2048, 0.5, False)])
def test_topk_from_scores_wan_bit_exact(dev, cols, ratio, ties):
    layout = ScoringLayout(cols * 128 - 7, cols * 128 - 7, 16)
    pol = wan_policy(layout, ratio)
    heads = 3
    scores = _random_scores(heads, pol.scored_rows, pol.k_blocks, cols, ties)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    col_idx, mask = ops.topk_from_scores(scores.to(dev), pol, row_ptr, want_mask=True)
    want = orc.mask_from_scores_wan(scores, ratio)
    assert torch.equal(mask.cpu().bool(), want)
    # CSR lists ascending columns of the same set
    got = ops.csr_to_mask(row_ptr, col_idx, heads, pol.q_blocks, pol.k_blocks).cpu()
    assert torch.equal(got, want)
    cols_np = col_idx.cpu().numpy().reshape(heads * pol.q_blocks, pol.k_pick)
    assert (np.diff(cols_np, axis=1) > 0).all()
    # the reference's literal torch.topk + scatter_ selects the same set on every
    # row where no tie straddles the k-th place
    clean = ~orc.boundary_ties(scores, pol.k_pick)
    assert torch.equal(want[clean], orc.mask_from_scores_torch(scores, pol.k_pick)[clean])


@pytest.mark.parametrize("video,text,ratio", [(118800, 256, 0.3), (1000, 60, 0.5),
                                              (1000, 0, 0.3), (1024, 0, 0.3), (3000, 256, 0.2)])
def test_topk_from_scores_hunyuan_policy(dev, video, text, ratio):
    layout = ScoringLayout(video + text, video, 16)
    pol = hunyuan_policy(layout, ratio)
    heads = 2
    scores = _random_scores(heads, pol.scored_rows, pol.k_blocks, video)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    col_idx, mask = ops.topk_from_scores(scores.to(dev), pol, row_ptr, want_mask=True)
    want = orc.mask_from_scores_hunyuan(scores, ratio, video + text, video)
    assert torch.equal(mask.cpu().bool(), want)
    assert torch.equal(ops.csr_to_mask(row_ptr, col_idx, heads, pol.q_blocks, pol.k_blocks).cpu(), want)


@pytest.mark.parametrize("d,tile,video,text,heads,k_tile", [
    (128, 16, 4 * 16 * 16, 0, 2, None), (128, 16, 3 * 20 * 21, 0, 2, None), (64, 16, 4 * 16 * 16, 0, 2, None),
    (128, 32, 2000, 0, 2, None), (128, 16, 2000, 100, 2, None), (64, 32, 1500, 100, 2, None),
    (128, 16, 20 * 128 + 16, 120, 2, None),  # last scored row dense, alone in its group
    (128, 16, 3000, 0, 8, None), (128, 16, 2000, 100, 16, None),  # heads divisible by 8: whole heads per XCD
    # the generic scorer: every other tile size, equal or not (attention_wan.py:94-95, 227-246)
    (128, 8, 2000, 0, 2, 8), (128, 64, 2000, 0, 2, 64), (128, 128, 2000, 100, 2, 128), (128, 4, 1000, 0, 2, 4),
    (128, 8, 2000, 0, 3, 64), (128, 64, 2000, 0, 2, 8), (128, 16, 2000, 100, 2, 32), (128, 32, 1500, 0, 2, 16),
    (64, 128, 1500, 100, 2, 4), (64, 4, 1000, 0, 2, 128), (128, 16, 2000, 100, 2, 8)])
def test_block_score_topk_matches_oracle(dev, d, tile, video, text, heads, k_tile):
    from dfsattn_amd.workloads import DfsConfig, synth_qkv
    cfg = DfsConfig("t", (1, 1, video), heads, d, torch.bfloat16, text_len=text, tile=tile, seed=3)
    q, k, v = synth_qkv(cfg)
    length = video + text
    print(f"scoring case d={d} tiles={tile}/{k_tile} video={video} text={text} heads={heads}", flush=True)
    perm, _ = orc.full_permutation(torch.randperm(video, generator=torch.Generator().manual_seed(5)), length)
    layout = ScoringLayout(length, video, tile, k_tile=k_tile)
    pol = wan_policy(layout, 0.3) if text == 0 else hunyuan_policy(layout, 0.3)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    prep = ops.prepare_qkv(q.to(dev), k.to(dev), v.to(dev), perm.to(dev, torch.int32), layout)
    col_idx, scores, mask = ops.block_score_topk(prep, pol, row_ptr, want_scores=True, want_mask=True)
    qp, kp = orc.apply_permutation(q, perm), orc.apply_permutation(k, perm)
    ref = orc.block_scores(qp, kp, tile, 128, video if text else None, k_tile=k_tile)
    got = scores.cpu()
    assert got.shape == ref.shape
    err = (got.double() - ref.double()).abs()
    print(f"  score error: max abs {float(err.max()):.3g}, max rel {float((err / ref.double().abs().clamp_min(1e-30)).max()):.3g},"
          f" max rel above 1e-3 {float((err / ref.double().abs())[ref > 1e-3].max()):.3g}", flush=True)
    # measured: at most 4e-7 relative on every entry (hi/lo-split products)
    assert torch.allclose(got, ref, rtol=1e-5, atol=1e-10), float((got - ref).abs().max())
    # every scored row of the block scores sums to block/tile
    assert torch.allclose(got.sum(-1), torch.full_like(got.sum(-1), 128 / tile), rtol=1e-4)
    # the fused top-k equals the oracle's selection on the same fp32 scores
    sel = orc.mask_from_scores_wan(got, 0.3) if text == 0 else \
        orc.mask_from_scores_hunyuan(got, 0.3, length, video)
    assert torch.equal(mask.cpu().bool(), sel)
    assert torch.equal(ops.csr_to_mask(row_ptr, col_idx, heads, pol.q_blocks, pol.k_blocks).cpu(), sel)
    # and agrees with the oracle's own fp32 mask wherever the k-th and
    # (k+1)-th oracle scores of a row are further apart than twice the
    # measured score error
    ref_sel = orc.mask_from_scores_wan(ref, 0.3) if text == 0 else \
        orc.mask_from_scores_hunyuan(ref, 0.3, length, video)
    err = float((got - ref).abs().max())
    for h in range(heads):
        for r in range(ref.shape[1]):
            if not torch.equal(sel[h, r], ref_sel[h, r]):
                top = torch.sort(ref[h, r, :pol.n_cand], descending=True).values
                assert float(top[pol.k_pick - 1] - top[pol.k_pick]) <= 2 * err, (h, r, err)


@pytest.mark.parametrize("video,text", [(4 * 16 * 16 * 4, 0), (2000, 100)])
def test_block_score_topk_lds_sums_path_selects_the_same(dev, video, text):
    """dfs_block_score_topk without a score matrix keeps its block sums in
    LDS; its selection equals the two-pass global-sums path's (the same
    arithmetic), and the one-pass path's scores agree with both to fp32
    rounding."""
    import ctypes
    from dfsattn_amd import _lib
    from dfsattn_amd.ops import _policy_args
    from dfsattn_amd.workloads import DfsConfig, synth_qkv
    heads = 3
    cfg = DfsConfig("t", (1, 1, video), heads, 128, torch.bfloat16, text_len=text, seed=6)
    q, k, v = synth_qkv(cfg)
    length = video + text
    perm, _ = orc.full_permutation(torch.randperm(video, generator=torch.Generator().manual_seed(2)), length)
    layout = ScoringLayout(length, video, 16)
    pol = wan_policy(layout, 0.3) if text == 0 else hunyuan_policy(layout, 0.3)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    prep = ops.prepare_qkv(q.to(dev), k.to(dev), v.to(dev), perm.to(dev, torch.int32), layout)
    col_global, scores2, _ = ops.block_score_topk(prep, pol, row_ptr, want_scores=True, one_pass=False)
    col_lds = torch.empty_like(col_global)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    _lib.call("dfs_block_score_topk", p(prep.q_hi), p(prep.q_lo), p(prep.k_hi), p(prep.k_lo), heads, 128, 16, 16,
              *_policy_args(pol), p(row_ptr), p(col_lds), None, None, None, 0,
              ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream))
    assert torch.equal(col_lds.cpu(), col_global.cpu())
    _, scores1, _ = ops.block_score_topk(prep, pol, row_ptr, want_scores=True, one_pass=True)
    torch.testing.assert_close(scores1.cpu(), scores2.cpu(), rtol=2e-5, atol=1e-7)


def test_block_score_topk_workspace_checks(dev):
    """The one-pass form needs a large enough, aligned workspace; the score
    matrix is optional there, and the selection is the same without it."""
    import ctypes
    from dfsattn_amd import _lib
    from dfsattn_amd.ops import _policy_args, score_workspace_bytes
    heads, length = 2, 1000
    q = torch.randn(1, heads, length, 64).bfloat16().to(dev)
    layout = ScoringLayout(length, length, 16)
    pol = wan_policy(layout, 0.3)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    prep = ops.prepare_qkv(q, q, q, torch.arange(length, dtype=torch.int32, device=dev), layout)
    need = score_workspace_bytes(heads, 16, 16, pol.q_blocks, pol.k_blocks)
    # rows of 16 query blocks per workgroup x 8 tiles, key blocks padded to 32-tile chunks
    assert need == heads * 16 * 8 * 8 * 4
    ws = torch.empty(need // 4 + 4, dtype=torch.float32, device=dev)
    col = torch.empty(pol.nnz(heads), dtype=torch.int32, device=dev)
    scores = torch.empty((heads, pol.scored_rows, pol.k_blocks), dtype=torch.float32, device=dev)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    stream = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    args = (p(prep.q_hi), p(prep.q_lo), p(prep.k_hi), p(prep.k_lo), heads, 64, 16, 16, *_policy_args(pol), p(row_ptr),
            p(col))
    for sc, w, nbytes in ((p(scores), p(ws), need - 4), (p(scores), ctypes.c_void_p(ws.data_ptr() + 4), need)):
        with pytest.raises(_lib.DfsKernelError):
            _lib.call("dfs_block_score_topk", *args, sc, None, w, nbytes, stream)
    _lib.call("dfs_block_score_topk", *args, p(scores), None, p(ws), need, stream)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(scores).all())
    with_scores = col.clone()
    col.fill_(-1)
    _lib.call("dfs_block_score_topk", *args, None, None, p(ws), need, stream)
    torch.cuda.synchronize()
    assert torch.equal(col, with_scores)


@pytest.mark.parametrize("heads,length,text", [(2, 3000, 0), (8, 2000, 0), (2, 2000, 100)])
def test_block_score_topk_all_tied_keeps_lowest_columns(dev, heads, length, text):
    """Q = 0 makes every logit 0, so every scored block sums exactly the same
    (its 64 tile pairs of 1/Z each): the top-k is one big tie, and the fused
    selection (one-pass and two-pass forms, whole heads per XCD at 8 heads)
    keeps the lowest candidate columns, as a stable descending sort does."""
    video = length - text
    q = torch.zeros(1, heads, length, 128, dtype=torch.bfloat16, device=dev)
    k = torch.randn(1, heads, length, 128, generator=torch.Generator().manual_seed(4)).bfloat16().to(dev)
    layout = ScoringLayout(length, video, 16)
    pol = wan_policy(layout, 0.3) if text == 0 else hunyuan_policy(layout, 0.3)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    prep = ops.prepare_qkv(q, k, k, torch.arange(length, dtype=torch.int32, device=dev), layout)
    want = torch.zeros((heads, pol.q_blocks, pol.k_blocks), dtype=torch.bool)
    want[:, :pol.dense_row, :pol.k_pick] = True
    want[:, :pol.dense_row, pol.dense_col:] = True
    want[:, pol.dense_row:] = True
    for one_pass in (True, False):
        _, scores, mask = ops.block_score_topk(prep, pol, row_ptr, want_scores=True, want_mask=True,
                                               one_pass=one_pass)
        got = scores.cpu()[:, :min(pol.scored_rows, pol.dense_row), :pol.n_cand]
        assert bool((got == got[0, 0, 0]).all())  # one tie over every candidate
        assert torch.equal(mask.cpu().bool(), want), one_pass


@pytest.mark.parametrize("d,tile,heads,video,text,q_size", [
    (128, 16, 2, 64 * 128, 0, 1.0),      # 64 columns: one register of keys
    (64, 16, 1, 64 * 128 + 5, 0, 1.0),   # 65 columns: four registers
    (128, 32, 3, 256 * 128, 0, 1.0),     # 256 columns, 8 rows per wave of the unsplit form
    (64, 32, 1, 257 * 128 - 3, 0, 1.0),  # 257 columns: radix selection
    (128, 16, 8, 2000, 100, 1.0),        # dense text rows and columns
    (128, 16, 1, 100, 0, 1.0),           # one block, one chunk
    (64, 16, 2, 3000, 0, 0.0),           # every score tied
    (128, 16, 2, 6000, 0, 40.0),         # logits far apart: shares with references far apart
])
def test_block_score_topk_split_matches_unsplit(dev, d, tile, heads, video, text, q_size):
    """Small problems divide the key chunks over workgroups and select in a
    second kernel: scores against the one-kernel form within fp32 rounding of
    sums in another order, and the selection of each form's own scores."""
    print(f"split d={d} tile={tile} heads={heads} video={video} text={text}", flush=True)
    L = video + text
    g = torch.Generator().manual_seed(L + tile)
    field = torch.randn((1, heads, -(-L // 96), d), generator=g).repeat_interleave(96, dim=2)[:, :, :L]
    q, k = (field + 0.5 * torch.randn((1, heads, L, d), generator=g) for _ in range(2))
    q, k = (q * q_size).to(torch.bfloat16).to(dev), k.to(torch.bfloat16).to(dev)
    layout = ScoringLayout(L, video, tile)
    pol = hunyuan_policy(layout, 0.5) if text else wan_policy(layout, 0.3)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    prep = ops.prepare_qkv(q, k, q, torch.arange(L, dtype=torch.int32, device=dev), layout)
    res = {}
    for split in (False, True):
        cols, scores, mask = ops.block_score_topk(prep, pol, row_ptr, want_scores=True, want_mask=True, split=split)
        only, _, _ = ops.block_score_topk(prep, pol, row_ptr, split=split)
        assert torch.equal(cols, only)  # asking for scores changes nothing
        sel = (orc.mask_from_scores_hunyuan(scores.cpu(), 0.5, L, video) if text
               else orc.mask_from_scores_wan(scores.cpu(), 0.3))
        assert torch.equal(mask.bool().cpu(), sel)
        back = ops.csr_to_mask(row_ptr, cols, heads, pol.q_blocks, pol.k_blocks)
        assert torch.equal(back, mask.bool())
        res[split] = scores.cpu()
    # sums of at most 2^8 terms per tile and of the shares in another order
    assert torch.allclose(res[True], res[False], rtol=1e-5, atol=1e-10)


@pytest.mark.parametrize("direction", ["rising", "falling"])
@pytest.mark.parametrize("tile,one_pass", [(16, True), (32, True), (16, False), (32, False)])
def test_block_scores_with_far_apart_logits(dev, direction, tile, one_pass):
    """Key tiles whose logits rise (or fall) by ~130 log2 units across the
    row: the scoring pass's reference (the first chunk's maximum) has to
    move for rising logits (in the one-pass form, rescaling the block sums
    already stored) and stays for falling ones; every form matches the fp32
    softmax of the oracle."""
    length, d = 2048, 128
    ramp = torch.linspace(0.0, 8.0, length)
    if direction == "falling":
        ramp = ramp.flip(0)
    q = torch.ones(1, 1, length, d).bfloat16()
    k = (ramp[None, None, :, None] * torch.ones(1, 1, length, d)).bfloat16()
    v = torch.zeros_like(q)
    layout = ScoringLayout(length, length, tile)
    pol = wan_policy(layout, 0.3)
    row_ptr = torch.from_numpy(pol.row_ptr(1)).to(dev)
    ident = torch.arange(length, dtype=torch.int32)
    prep = ops.prepare_qkv(q.to(dev), k.to(dev), v.to(dev), ident.to(dev), layout)
    _, scores, _ = ops.block_score_topk(prep, pol, row_ptr, want_scores=True, one_pass=one_pass)
    ref = orc.block_scores(q.float(), k.float(), tile, 128, None)
    got = scores.cpu()
    assert bool(torch.isfinite(got).all())
    err = (got.double() - ref.double()).abs()
    print(f"far-apart logits {direction} tile={tile} one_pass={one_pass}: max abs {float(err.max()):.3g}, "
          f"max rel above 1e-6 {float((err / ref.double().abs())[ref > 1e-6].max()):.3g}", flush=True)
    assert torch.allclose(got, ref, rtol=1e-4, atol=1e-9), float((got - ref).abs().max())


def _run_bsa(dev, q, k, v, mask_bool, pv, out_dtype, perm=None, scale=None):
    heads, length, d = q.shape[1], q.shape[2], q.shape[3]
    layout = ScoringLayout(length, length, 16)
    ident = torch.arange(length, dtype=torch.int32)
    prep = ops.prepare_qkv(q.to(dev), k.to(dev), v.to(dev), ident.to(dev), layout, operand_dtype=pv, pool=False)
    row_ptr, col_idx = ops.mask_to_csr(mask_bool.to(dev))
    out = ops.bsa_fwd(prep, row_ptr, col_idx, out_dtype=out_dtype, scale=scale,
                      out_perm=None if perm is None else perm.to(dev, torch.int32))
    return out.cpu()


SCALES = (None, 0.6)  # the softmax scale: default D^-1/2, and one that sends every head to the scaled instance


@pytest.mark.parametrize("scale", SCALES)
@pytest.mark.parametrize("d,length,density,pv", [
    (128, 1000, 0.3, torch.float16), (128, 1024, 0.5, torch.float16), (64, 1000, 0.3, torch.float16),
    (128, 3000, 0.3, torch.float16), (128, 1000, 1.0, torch.float16), (128, 1000, 0.3, torch.bfloat16),
    (64, 130, 1.0, torch.float16), (128, 1100, 0.3, torch.float16), (64, 1400, 0.2, torch.bfloat16)])
def test_bsa_fwd_matches_masked_dense(dev, scale, d, length, density, pv):
    """The attention kernel against fp32 masked attention, at the default
    softmax scale and at one large enough that every head runs in the scaled
    instance (rows carrying their own powers of two)."""
    from dfsattn_amd.workloads import DfsConfig, synth_qkv
    heads = 2
    cfg = DfsConfig("t", (1, 1, length), heads, d, torch.bfloat16, seed=11)
    q, k, v = synth_qkv(cfg)
    nb = math.ceil(length / 128)
    g = torch.Generator().manual_seed(12)
    mask = torch.rand((heads, nb, nb), generator=g) < density
    mask[:, torch.arange(nb), torch.arange(nb)] = True  # no empty rows
    out = _run_bsa(dev, q, k, v, mask, pv, torch.float32, scale=scale)
    ref = orc.masked_attention(q, k, v, mask, scale=scale)
    max_abs = float((out - ref).abs().max())
    mr = mean_rel(out, ref)
    tol = 1e-3 if pv == torch.float16 else 3e-3  # bf16 P: reference-kernel precision class
    assert max_abs <= 2e-2 and mr <= tol, (max_abs, mr)
    if density == 1.0:
        dense = orc.dense_attention(q, k, v, scale=scale)
        assert mean_rel(out, dense) <= tol


@pytest.mark.parametrize("length", [127, 129, 255, 257, 383, 641])
@pytest.mark.parametrize("heads,d", [(1, 128), (3, 64), (5, 128)])
def test_bsa_fwd_ragged_lengths(dev, length, heads, d):
    """Lengths just under and over multiples of the 128-token block (the
    last block's keys masked, its rows dropped) with odd head counts, at the
    output contract on fp32 output."""
    from dfsattn_amd.workloads import DfsConfig, synth_qkv
    cfg = DfsConfig("t", (1, 1, length), heads, d, torch.bfloat16, seed=length + heads)
    q, k, v = synth_qkv(cfg)
    nb = math.ceil(length / 128)
    mask = torch.rand((heads, nb, nb), generator=torch.Generator().manual_seed(length)) < 0.5
    mask[:, :, nb - 1] = True  # every row sees the partial block
    out = _run_bsa(dev, q, k, v, mask, torch.float16, torch.float32)
    ref = orc.masked_attention(q, k, v, mask)
    assert out.shape == ref.shape
    assert float((out - ref).abs().max()) <= 2e-2 and mean_rel(out, ref) <= 1e-3


def test_bsa_fwd_bf16_out_and_fused_unpermute(dev):
    from dfsattn_amd.workloads import DfsConfig, synth_qkv
    heads, d, length = 2, 128, 1000
    cfg = DfsConfig("t", (1, 1, length), heads, d, torch.bfloat16, seed=13)
    q, k, v = synth_qkv(cfg)
    nb = math.ceil(length / 128)
    mask = torch.rand((heads, nb, nb), generator=torch.Generator().manual_seed(2)) < 0.4
    mask[:, :, 0] = True
    perm = torch.randperm(length, generator=torch.Generator().manual_seed(3))
    out32 = _run_bsa(dev, q, k, v, mask, torch.float16, torch.float32)
    out16 = _run_bsa(dev, q, k, v, mask, torch.float16, torch.bfloat16)
    assert torch.equal(out16, out32.to(torch.bfloat16))
    scat = _run_bsa(dev, q, k, v, mask, torch.float16, torch.float32, perm=perm)
    assert torch.equal(scat[:, :, perm], out32)


@pytest.mark.parametrize("scale", SCALES)
def test_empty_rows_give_zero(dev, scale):
    heads, d, length = 1, 128, 512
    q, k, v = (torch.randn((1, heads, length, d)).to(torch.bfloat16) for _ in range(3))
    mask = torch.zeros((heads, 4, 4), dtype=torch.bool)
    mask[0, 0, 1] = True
    out = _run_bsa(dev, q, k, v, mask, torch.float16, torch.float32, scale=scale)
    assert torch.count_nonzero(out[:, :, 128:]) == 0
    ref = orc.masked_attention(q, k, v, mask, scale=scale)
    assert mean_rel(out[:, :, :128], ref[:, :, :128]) < 1e-3


@pytest.mark.parametrize("scale", SCALES)
def test_rows_keeping_only_a_short_tail_block(dev, scale):
    """The last block holds 26 keys: a wave whose keys of that block are all
    masked, and which has seen no other key, must contribute nothing."""
    heads, d, length = 2, 128, 1050
    q, k, v = (torch.randn((1, heads, length, d), generator=torch.Generator().manual_seed(s)).to(torch.bfloat16)
               for s in (21, 22, 23))
    nb = math.ceil(length / 128)
    mask = torch.rand((heads, nb, nb), generator=torch.Generator().manual_seed(24)) < 0.3
    mask[:, 0] = False
    mask[:, 0, nb - 1] = True   # only the tail block
    mask[:, 1] = False
    mask[:, 1, 3] = True
    mask[:, 1, nb - 1] = True
    mask[:, nb - 1] = False
    mask[:, nb - 1, nb - 1] = True
    out = _run_bsa(dev, q, k, v, mask, torch.float16, torch.float32, scale=scale)
    assert torch.isfinite(out).all()
    ref = orc.masked_attention(q, k, v, mask, scale=scale)
    assert float((out - ref).abs().max()) <= 2e-2 and mean_rel(out, ref) <= 1e-3


@pytest.mark.parametrize("scale", SCALES)
def test_bsa_fwd_rising_and_negative_logits(dev, scale):
    """Logits that grow block after block (the running maximum jumps by far
    more than the lazy-rescale threshold several times) and rows whose
    logits are all strongly negative: the output still equals fp32 masked
    attention."""
    heads, d, length = 2, 128, 1200
    g = torch.Generator().manual_seed(21)
    q = torch.randn((1, heads, length, d), generator=g)
    k = torch.randn((1, heads, length, d), generator=g)
    v = torch.randn((1, heads, length, d), generator=g)
    nb = math.ceil(length / 128)
    ramp = torch.linspace(0.2, 3.0, nb).repeat_interleave(128)[:length]
    k = k * ramp[None, None, :, None]          # later key blocks give much larger |logits|
    q[:, 1] = -q[:, 1].abs()                   # head 1: many large negative logits
    k[:, 1] = k[:, 1].abs()
    q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    mask = torch.rand((heads, nb, nb), generator=g) < 0.6
    mask[:, torch.arange(nb), torch.arange(nb)] = True
    out = _run_bsa(dev, q, k, v, mask, torch.float16, torch.float32, scale=scale)
    ref = orc.masked_attention(q, k, v, mask, scale=scale)
    assert torch.isfinite(out).all()
    assert float((out - ref).abs().max()) <= 2e-2 and mean_rel(out, ref) <= 1e-3, \
        (float((out - ref).abs().max()), mean_rel(out, ref))


@pytest.mark.parametrize("d,length,scale,v_size", [(128, 1200, None, 1.0), (64, 641, None, 1e30), (128, 385, 0.6, 1.0)])
def test_bsa_fwd_bf16_operands_moving_reference(dev, d, length, scale, v_size):
    """bf16 operands, whose scores stay in units of q.k: block maxima that
    rise from block to block, so the reference moves; V far beyond f16."""
    heads = 2
    g = torch.Generator().manual_seed(27)
    q, k, v = (torch.randn((1, heads, length, d), generator=g) for _ in range(3))
    nb = math.ceil(length / 128)
    k = k * torch.linspace(0.2, 4.0, nb).repeat_interleave(128)[:length][None, None, :, None]
    q[:, 1], k[:, 1] = -q[:, 1].abs(), k[:, 1].abs()  # head 1: large negative logits
    q, k, v = q.to(torch.bfloat16), k.to(torch.bfloat16), (v * v_size).to(torch.bfloat16)
    mask = torch.rand((heads, nb, nb), generator=g) < 0.6
    mask[:, torch.arange(nb), torch.arange(nb)] = True
    out = _run_bsa(dev, q, k, v, mask, torch.bfloat16, torch.float32, scale=scale)
    ref = orc.masked_attention(q, k, v, mask, scale=scale)
    assert torch.isfinite(out).all()
    # P is rounded to bf16 (2^-9 each): the class tolerance of the shape test
    assert mean_rel(out, ref) <= 3e-3, mean_rel(out, ref)
    assert float((out - ref).abs().max()) <= 2e-2 * v_size


@pytest.mark.parametrize("d,heads,video,text,cut,dtype,out_dtype,plan", [
    (128, 3, 1300, 0, None, torch.bfloat16, torch.float32, (1, 0, 3, 8)),   # every block in 3 parts, a ragged last one
    (64, 2, 2000, 0, None, torch.float16, torch.bfloat16, (1, 3, 2, 4)),    # the tail of each XCD's list
    (128, 2, 1024, 200, None, torch.bfloat16, torch.bfloat16, (4, 0, 1, 1)),  # long rows in parts, the rest whole
    (128, 1, 1152, 150, 1200, torch.bfloat16, torch.float32, (8, 1, 5, 2)),   # both, with a second sequence
    (64, 3, 300, 0, None, torch.bfloat16, torch.float32, (1, 0, 64, 1)),    # more parts than columns: empty parts
    (128, 2, 1000, 0, 700, torch.bfloat16, torch.float16, (1, 0, 4, 4)),    # whole query blocks past the first sequence
])
def test_bsa_fwd_parts_match_unsplit(dev, monkeypatch, d, heads, video, text, cut, dtype, out_dtype, plan):
    """Query blocks cut into parts (long_parts, full_rows, parts) and dealt in
    other ranges (chunks) against the same call uncut: the sums run
    in another order (and P is rounded against another reference), nothing
    else changes. Head 0 holds a value beyond f16, so its blocks run whole in
    the scaled instance beside the cut ones."""
    print(f"parts d={d} heads={heads} video={video} text={text} cut={cut} plan={plan}", flush=True)
    L = video + text
    g = torch.Generator().manual_seed(L + d)
    q, k, v = (torch.randn((1, heads, L, d), generator=g).to(dtype) for _ in range(3))
    if dtype == torch.bfloat16:
        q[0, 0, 5, 3] = 1.0e5
        k[0, 0, 5, 3] = 0.0
    layout = ScoringLayout(L, video, 16)
    perm = torch.randperm(L, generator=g).to(torch.int32)
    mask = torch.rand((heads, layout.q_blocks, layout.k_blocks), generator=g) < 0.5
    mask[:, 0] = False  # empty rows
    mask[:, video // 128:] = True
    mask[:, 1] = False
    mask[:, 1, -1] = True  # one column: most parts empty
    prep = ops.prepare_qkv(*(x.to(dev) for x in (q, k, v)), perm.to(dev), layout, pool=False, q_operand=False)
    row_ptr, col_idx = ops.mask_to_csr(mask.to(dev))
    cu = None if cut is None else torch.tensor([0, cut, L], dtype=torch.int32, device=dev)
    got = {}
    for name, pl in (("whole", (1, 0, 1, 8)), ("parts", plan)):
        monkeypatch.setattr(ops, "query_plan", lambda lay, *a: (lay.video_len // 128 if lay.text_len else lay.q_blocks, *pl))
        got[name] = ops.bsa_fwd(prep, row_ptr, col_idx, out_dtype=out_dtype, out_perm=perm.to(dev), want_lse=True,
                                cu_seqlens_q=cu, cu_seqlens_k=cu)
    (o0, l0), (o1, l1) = ((o.float().cpu(), l.cpu()) for o, l in (got["whole"], got["parts"]))
    assert torch.equal(torch.isinf(l0), torch.isinf(l1))
    fin = torch.isfinite(l0)
    # l sums f16-rounded P (2^-11 each, against another power-of-two-free
    # reference per part): relative 2^-11 at most, so lse within 2^-11 absolute
    assert float((l0 - l1)[fin].abs().max()) <= 2.0 ** -11 + 2e-6 * float(l0[fin].abs().max())
    if dtype == torch.bfloat16:
        assert torch.equal(o0[0, 0], o1[0, 0])  # the scaled head is never cut
    rel = float((o0 - o1).norm() / o0.norm())
    ulp = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[out_dtype]
    assert rel <= 2.0 ** -11 + ulp, rel  # P's rounding, averaged over the keys, and the output's
    assert float((o0 - o1).abs().max()) <= 1e-2


@pytest.mark.parametrize("value", [math.nan, math.inf, -math.inf])
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("d,heads,video,text,dtype,plan", [
    (128, 2, 1300, 0, torch.bfloat16, (1, 0, 3, 4)),    # every block in 3 parts
    (64, 1, 2000, 0, torch.float16, (1, 1, 2, 8)),      # the tail of each XCD's list
    (128, 1, 1024, 200, torch.bfloat16, (4, 0, 1, 8)),  # long rows in parts, the rest whole
])
def test_bsa_fwd_parts_keep_nan(dev, monkeypatch, d, heads, video, text, dtype, plan, where, value):
    """One NaN or infinity in Q, K or V shows in the same rows whether their
    query blocks are cut or not."""
    print(f"parts d={d} heads={heads} video={video} text={text} plan={plan} {where}={value}", flush=True)
    L = video + text
    g = torch.Generator().manual_seed(L)
    x = {n: torch.randn((1, heads, L, d), generator=g).to(dtype) for n in "qkv"}
    x[where][0, heads - 1, 1030, 3] = value
    layout = ScoringLayout(L, video, 16)
    mask = torch.rand((heads, layout.q_blocks, layout.k_blocks), generator=g) < 0.5
    mask[:, video // 128:] = True
    mask[:, 0] = False  # an empty row
    prep = ops.prepare_qkv(*(x[n].to(dev) for n in "qkv"), torch.arange(L, dtype=torch.int32, device=dev), layout,
                           pool=False, q_operand=False)
    row_ptr, col_idx = ops.mask_to_csr(mask.to(dev))
    got = []
    for pl in ((1, 0, 1, 8), plan):
        monkeypatch.setattr(ops, "query_plan", lambda lay, *a: (lay.video_len // 128 if lay.text_len else lay.q_blocks, *pl))
        got.append([t.cpu() for t in ops.bsa_fwd(prep, row_ptr, col_idx, out_dtype=torch.float32, want_lse=True)])
    (o0, l0), (o1, l1) = got
    assert not torch.isfinite(o0).all()
    if where == "v":  # infinite or NaN, as P of the key is above or rounds to 0 against either reference
        assert torch.equal(torch.isfinite(o0), torch.isfinite(o1))
    else:
        assert torch.equal(torch.isnan(o0), torch.isnan(o1)) and not torch.isinf(o1).any()
    assert torch.equal(torch.isfinite(l0), torch.isfinite(l1))


@pytest.mark.parametrize("d,heads,video,text,tile,dtype,operand,big", [
    (128, 2, 1000, 0, 16, torch.bfloat16, None, ("k", 999)),   # one launch for q, k and v; flag in the last wave
    (64, 3, 1153, 0, 32, torch.bfloat16, None, ("v", 1152)),   # two V blocks per workgroup, an odd block count
    (128, 1, 900, 125, 16, torch.bfloat16, None, ("q", 0)),    # text; only Q beyond f16
    (128, 40, 3000, 0, 16, torch.bfloat16, None, ("v", 0)),    # above the one-launch limit
    (64, 2, 4000, 0, 16, torch.bfloat16, None, ("q", 3999)),   # a given mask: the attention marks the head itself
    (128, 3, 600, 0, 16, torch.bfloat16, None, ("q", 130, 1.0e5)),  # beyond f16, but not times the scale
    (64, 2, 500, 0, 16, torch.float16, None, None),            # nothing to flag
    (128, 2, 700, 0, 16, torch.bfloat16, torch.bfloat16, ("v", 5)),  # bf16 operands: no flags
    (128, 2, 700, 0, 64, torch.bfloat16, None, None),          # tiles of the generic scorer (score matrix)
])
def test_whole_call_matches_single_entry_points(dev, d, heads, video, text, tile, dtype, operand, big):
    """dfs_call (all phases at once, then one by one, and with a given mask)
    against prepare_qkv, block_score_topk and bsa_fwd: the same kernels on the
    same values, so the same columns and bits."""
    print(f"call d={d} heads={heads} video={video} text={text} tile={tile} {dtype} {operand} {big}", flush=True)
    L = video + text
    g = torch.Generator().manual_seed(L)
    x = {n: torch.randn((1, heads, L, d), generator=g).to(dtype) for n in "qkv"}
    if big:
        x[big[0]][0, heads - 1, big[1], d - 1] = big[2] if len(big) > 2 else 1.0e6
    q, k, v = (x[n].to(dev) for n in "qkv")
    layout = ScoringLayout(L, video, tile)
    pol = hunyuan_policy(layout, 0.5) if text else wan_policy(layout, 0.3)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    perm = torch.randperm(video, generator=g)
    perm = torch.cat([perm, torch.arange(video, L)]).to(torch.int32).to(dev)
    prep = ops.prepare_qkv(q, k, v, perm, layout, operand_dtype=operand, q_operand=False)
    cols, _, _ = ops.block_score_topk(prep, pol, row_ptr)
    ref = ops.bsa_fwd(prep, row_ptr, cols, out_perm=perm)
    kw = dict(operand_dtype=operand, out_perm=perm)
    call = ops.Call(q, k, v, perm, layout, pol, row_ptr, None, **kw)
    call.run()
    steps = ops.Call(q, k, v, perm, layout, pol, row_ptr, None, **kw)
    for phase in (ops.PREPARE, ops.SELECT, ops.ATTEND):
        steps.run(phase)
    given = ops.Call(q, k, v, perm, layout, pol, row_ptr, cols, **kw)
    given.run()
    assert torch.equal(call.col_idx, cols) and torch.equal(steps.col_idx, cols)
    for c in (call, steps, given):
        assert torch.equal(c.out, ref)


@pytest.mark.parametrize("d,video,text,cut,plan", [
    (128, 1300, 0, None, (1, 0, 1, 8)),    # uncut: the marked blocks alone are redone
    (64, 1300, 0, None, (1, 0, 3, 4)),     # every block in parts
    (128, 2000, 0, None, (1, 2, 2, 8)),    # the tail of each XCD's list in parts
    (128, 1024, 200, None, (4, 0, 1, 8)),  # the text rows in parts
    (128, 1024, 200, 1190, (4, 1, 2, 4)),  # both, with a second sequence
])
@pytest.mark.parametrize("rows", [(5,), (0, 700, 1023), "all", "inf"])
def test_call_redoes_blocks_with_q_beyond_f16(dev, monkeypatch, d, video, text, cut, plan, rows):
    """A given mask's call finds the rows of Q beyond f16 in the attention
    itself and does their query blocks again in the scaled instance: the bits
    of the separate calls, whose preparation finds the head and gives the
    scaled instance all of it."""
    L, heads = video + text, 2
    print(f"q beyond f16 d={d} video={video} text={text} cut={cut} plan={plan} rows={rows}", flush=True)
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn((1, heads, L, d), generator=g).to(torch.bfloat16) for _ in range(3))
    if rows == "inf":  # not beyond the range: it stays what it is in either instance
        q[0, 1, 300, 3], q[0, 1, 301, 4] = math.inf, math.nan
    else:
        q[0, 1, slice(None) if rows == "all" else list(rows), 3] = 1.0e6
    q, k, v = (t.to(dev) for t in (q, k, v))
    layout = ScoringLayout(L, video, 16)
    pol = hunyuan_policy(layout, 0.6) if text else wan_policy(layout, 0.4)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    perm = torch.cat([torch.randperm(video, generator=g), torch.arange(video, L)]).to(torch.int32).to(dev)
    cu = None if cut is None else torch.tensor([0, cut, L], dtype=torch.int32, device=dev)
    prep = ops.prepare_qkv(q, k, v, perm, layout, q_operand=False)
    cols, _, _ = ops.block_score_topk(prep, pol, row_ptr)
    long_row = video // 128 if text else layout.q_blocks
    monkeypatch.setattr(ops, "query_plan", lambda *a: (long_row, 1, 0, 1, 8))
    ref = ops.bsa_fwd(prep, row_ptr, cols, out_perm=perm, cu_seqlens_q=cu, cu_seqlens_k=cu)
    monkeypatch.setattr(ops, "query_plan", lambda *a: (long_row, *plan))
    ops._call_template.cache_clear()
    try:
        call = ops.Call(q, k, v, perm, layout, pol, row_ptr, cols, out_perm=perm, cu_seqlens_q=cu, cu_seqlens_k=cu)
        for _ in range(2):  # the marks of the first run are cleared
            call.run()
            got, want = call.out.nan_to_num(nan=7.0), ref.nan_to_num(nan=7.0)
            if plan == (1, 0, 1, 8):
                assert torch.equal(got, want)
            elif rows == "inf":
                assert torch.equal(call.out.isnan(), ref.isnan())
            else:
                assert torch.equal(got[0, 1], want[0, 1])
    finally:
        ops._call_template.cache_clear()


@pytest.mark.parametrize("d,heads,L,cut,layouts,big", [
    (128, 3, 1000, None, ("token", "token", "token"), None),
    (64, 2, 700, None, ("head", "slice", "token"), None),
    (128, 2, 900, 800, ("token", "head", "slice"), "v"),   # a second sequence; V beyond f16 rewritten by the fix-up
    (128, 2, 520, None, ("slice", "token", "head"), "k"),
    (64, 1, 300, None, ("token", "odd", "token"), "q"),    # one head; rows off 16 bytes are copied
])
@pytest.mark.parametrize("given", [False, True])
def test_call_reads_strided_inputs(dev, d, heads, L, cut, layouts, big, given):
    """q, k and v as views of [L, H, D] storage, of a wider buffer, or with
    rows off the 16-byte boundary: the same columns and bits as contiguous
    inputs; the output is contiguous unless token order is asked for."""
    print(f"strided d={d} heads={heads} L={L} cut={cut} {layouts} big={big} given={given}", flush=True)
    g = torch.Generator().manual_seed(L + d)
    x = [torch.randn((1, heads, L, d), generator=g).to(torch.bfloat16).to(dev) for _ in range(3)]
    if big:
        x["qkv".index(big)][0, heads - 1, L - 1, 0] = 1.0e6
    layout = ScoringLayout(L, L, 16)
    pol = wan_policy(layout, 0.4)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    perm = torch.randperm(L, generator=g).to(torch.int32).to(dev)
    cu = None if cut is None else torch.tensor([0, cut, L], dtype=torch.int32, device=dev)
    kw = dict(out_perm=perm, cu_seqlens_q=cu, cu_seqlens_k=cu)

    def view(t, how):
        if how == "token":
            return t.transpose(1, 2).contiguous().transpose(1, 2)
        if how == "head":
            return t
        pad = 8 if how == "slice" else 1  # a row pitch of D + 8 elements, or of D + 1 on odd bases
        buf = torch.zeros((1, heads, L, d + pad), dtype=t.dtype, device=dev)
        buf[..., pad:] = t
        return buf[..., pad:]

    ref = ops.Call(*x, perm, layout, pol, row_ptr, None, **kw)
    ref.run()
    got = ops.Call(*(view(t, how) for t, how in zip(x, layouts)), perm, layout, pol, row_ptr,
                   ref.col_idx if given else None, token_major=given, **kw)
    got.run()
    assert torch.equal(got.col_idx, ref.col_idx) and torch.equal(got.out, ref.out)
    assert got.out.shape == ref.out.shape and (got.out.transpose(1, 2) if given else got.out).is_contiguous()


def _running_maximum_rows(q, k, v, scale):
    """One head in 64 bits with P rounded to bf16 against the running maximum,
    key blocks in the kernel's order (distance from the query block)."""
    L, nb = q.shape[0], math.ceil(q.shape[0] / 128)
    s = (q @ k.t()) * (scale * math.log2(math.e))
    out = torch.empty_like(q)
    for qb in range(nb):
        rows = slice(128 * qb, min(128 * (qb + 1), L))
        m, l, o = torch.full((1, 1), -math.inf, dtype=torch.float64), 0.0, 0.0
        for c in sorted(range(nb), key=lambda c: 2 * abs(c - qb) + (c > qb)):
            keys = slice(128 * c, min(128 * (c + 1), L))
            mn = torch.maximum(m, s[rows, keys].amax(1, keepdim=True))
            p, a = torch.exp2(s[rows, keys] - mn).float().bfloat16().double(), torch.exp2(m - mn)
            m, l, o = mn, l * a + p.sum(1, keepdim=True), o * a + p @ v[keys]
        out[rows] = o / l
    return out


@pytest.mark.parametrize("d,heads,length", [(128, 2, 1111), (64, 2, 1500)])
@pytest.mark.parametrize("parts", [False, True])
def test_bsa_fwd_bf16_operands_error_of_running_maximum(dev, monkeypatch, d, heads, length, parts):
    """The distance from 64-bit results is that of P rounded to bf16 against
    the running maximum: within 1% (fp32 sums, 2^-24 each, are far below; rows
    of other summation orders differ by far less than the 2.5 to 7% that a
    reference fixed at the first block costs). Cut into parts, each with its
    own maximum: 3% over the few hundred thousand values."""
    print(f"bf16 operands d={d} heads={heads} length={length} parts={parts}", flush=True)
    g = torch.Generator().manual_seed(length)
    q, k, v = (torch.randn((1, heads, length, d), generator=g).to(torch.bfloat16) for _ in range(3))
    nb = math.ceil(length / 128)
    plan = (nb, 1, 0, 3, 8) if parts else (nb, 1, 0, 1, 8)
    monkeypatch.setattr(ops, "query_plan", lambda *a: plan)
    out = _run_bsa(dev, q, k, v, torch.ones((heads, nb, nb), dtype=torch.bool), torch.bfloat16, torch.float32)
    err = ref_err = 0.0
    for h in range(heads):
        qh, kh, vh = (t[0, h].double() for t in (q, k, v))
        exact = torch.softmax(qh @ kh.t() / math.sqrt(d), -1) @ vh
        err += float((out[0, h].double() - exact).pow(2).sum())
        ref_err += float((_running_maximum_rows(qh, kh, vh, 1 / math.sqrt(d)) - exact).pow(2).sum())
    ratio = math.sqrt(err / ref_err)
    print(f"error over the running maximum's: {ratio:.4f}", flush=True)
    assert ratio <= (1.03 if parts else 1.01), ratio


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("parts", [1, 3])
def test_bsa_fwd_bf16_operands_large_v(dev, monkeypatch, d, parts):
    """V of 1e36, so that a block of 128 full weights just stays inside fp32,
    and key blocks that hold one weight 2^14 above those of the row's first
    block: P is at most 1, and O stays inside fp32 too."""
    L = 512
    g = torch.Generator().manual_seed(5)
    q = torch.zeros(1, 1, L, d)
    q[..., 0] = math.sqrt(d)
    k = 0.1 * torch.randn(1, 1, L, d, generator=g)
    k[0, 0, 133::128, 0] = 10.0
    v = (0.5 + torch.rand(1, 1, L, d, generator=g)) * 1e36
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    monkeypatch.setattr(ops, "query_plan", lambda *a: (4, 1, 0, parts, 8))
    out = _run_bsa(dev, q, k, v, torch.ones((1, 4, 4), dtype=torch.bool), torch.bfloat16, torch.float32)
    qh, kh, vh = (t[0, 0].double() for t in (q, k, v))
    ref = torch.softmax(qh @ kh.t() / math.sqrt(d), -1) @ vh
    assert torch.isfinite(out).all()
    assert mean_rel(out[0, 0], ref) <= 3e-3  # P rounded to bf16 (2^-9 each)


def test_wrappers_reject_bad_index_operands(dev):
    """Index operands must be contiguous int32 on the operands' device, and
    CSR offsets must cover every (head, query block) row: checked on the host
    before any launch."""
    length, heads = 300, 2
    q = torch.randn(1, heads, length, 64).bfloat16().to(dev)
    layout = ScoringLayout(length, length, 16)
    ident = torch.arange(length, dtype=torch.int32, device=dev)
    with pytest.raises(ValueError):
        ops.prepare_qkv(q, q, q, ident.long(), layout)
    with pytest.raises(ValueError):
        ops.permute_gather(q, ident.long())
    prep = ops.prepare_qkv(q, q, q, ident, layout)
    pol = wan_policy(layout, 0.5)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    col_idx, _, _ = ops.block_score_topk(prep, pol, row_ptr)
    with pytest.raises(ValueError):
        ops.bsa_fwd(prep, row_ptr.long(), col_idx)
    with pytest.raises(ValueError):
        ops.bsa_fwd(prep, row_ptr[:-1].contiguous(), col_idx)
    with pytest.raises(ValueError):
        ops.bsa_fwd(prep, row_ptr, col_idx, out_perm=ident.long())
    with pytest.raises(ValueError):
        ops.block_score_topk(prep, pol, row_ptr[1:].contiguous())
    with pytest.raises(ValueError):
        ops.csr_to_mask(row_ptr, col_idx.long(), heads, pol.q_blocks, pol.k_blocks)
    with pytest.raises(RuntimeError):
        ops.bsa_fwd(prep, row_ptr.cpu(), col_idx)
    # the valid call still runs after the rejections
    out = ops.bsa_fwd(prep, row_ptr, col_idx, out_perm=ident)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out.float()).all())


def test_call_rejects_bad_output_permutations(dev):
    """The call checks out_perm's place, type and length before it takes the
    address, and holds it until its launches are enqueued."""
    import gc
    import weakref
    length, heads = 300, 2
    q = torch.randn(1, heads, length, 64).bfloat16().to(dev)
    layout = ScoringLayout(length, length, 16)
    pol = wan_policy(layout, 0.5)
    row_ptr = torch.from_numpy(pol.row_ptr(heads)).to(dev)
    ident = torch.arange(length, dtype=torch.int32, device=dev)
    for bad, error in ((ident[:-1], ValueError), (ident.long(), ValueError), (ident.cpu(), RuntimeError)):
        with pytest.raises(error):
            ops.Call(q, q, q, ident, layout, pol, row_ptr, None, out_perm=bad)
    own = ident.clone()
    call, held = ops.Call(q, q, q, ident, layout, pol, row_ptr, None, out_perm=own), weakref.ref(own)
    del own
    gc.collect()
    assert held() is not None
    call.run()
    assert bool(torch.isfinite(call.out.float()).all())


@pytest.mark.parametrize("length,cu_q,cu_k", [
    (1300, [0, 1100, 1300], [0, 1100, 1300]),   # text padding: two sequences, blocks from each start
    (1300, [0, 1152, 1300], [0, 1152, 1300]),   # a split on a block boundary
    (1000, [0, 130, 1000], [0, 130, 1000]),     # a long second sequence
    (1000, [0, 1, 1000], [0, 1, 1000]),         # a one-token first sequence
    (1000, [0, 1000, 1000], [0, 700, 1000]),    # Wan's [0, S, S] / [0, s_k, S]: keys past s_k unused
    (1000, [0, 600, 900], [0, 500, 1000]),      # unequal splits; rows 900.. in no sequence
    (1000, [0, 1000], [0, 1000]),               # one sequence given explicitly
    (900, [0, 0, 900], [0, 0, 900]),            # an empty first sequence
])
def test_bsa_fwd_varlen_matches_oracle(dev, length, cu_q, cu_k):
    """Device cu_seqlens (block_sparse_attn_func's varlen arguments): sequence
    i's queries attend its keys under the mask indexed from each sequence's
    start; rows in no query sequence are zero; the offsets are never read on
    the host. Against the fp32 varlen oracle, which tests pin to dense
    attention under explicit token masks."""
    from dfsattn_amd.workloads import DfsConfig, synth_qkv
    heads, d = 2, 128
    cfg = DfsConfig("t", (1, 1, length), heads, d, torch.bfloat16, seed=21)
    q, k, v = synth_qkv(cfg)
    nb = math.ceil(length / 128)
    g = torch.Generator().manual_seed(22)
    mask = torch.rand((heads, nb, nb), generator=g) < 0.4
    mask[:, torch.arange(nb), torch.arange(nb)] = True
    layout = ScoringLayout(length, length, 16)
    ident = torch.arange(length, dtype=torch.int32)
    prep = ops.prepare_qkv(q.to(dev), k.to(dev), v.to(dev), ident.to(dev), layout, pool=False)
    row_ptr, col_idx = ops.mask_to_csr(mask.to(dev))
    out = torch.full((1, heads, length, d), 7.0, dtype=torch.float32, device=dev)
    cq = torch.tensor(cu_q, dtype=torch.int32, device=dev)
    ck = torch.tensor(cu_k, dtype=torch.int32, device=dev)
    _, lse = ops.bsa_fwd(prep, row_ptr, col_idx, out_dtype=torch.float32, out=out, cu_seqlens_q=cq,
                         cu_seqlens_k=ck, want_lse=True)
    got = out.cpu()
    ref = orc.varlen_attention(q, k, v, mask, cu_q, cu_k)
    assert float((got - ref).abs().max()) <= 2e-2 and mean_rel(got, ref) <= 1e-3
    covered = torch.zeros(length, dtype=torch.bool)
    for (q0, q1), (k0, k1) in zip(zip(cu_q, cu_q[1:]), zip(cu_k, cu_k[1:])):
        if k1 > k0:
            covered[q0:q1] = True
    assert bool((got[:, :, ~covered] == 0).all())
    assert bool(torch.isneginf(lse.cpu()[:, ~covered]).all())
    assert bool(torch.isfinite(lse.cpu()[:, covered]).all())


@pytest.mark.parametrize("length,cu_q,cu_k,far_rows", [
    (1000, [0, 1000, 1000], [0, 300, 1000], True),   # some rows keep only key blocks past cu_k[1]
    (1000, [0, 600, 1000], [0, 0, 1000], False),     # a first sequence with queries and no keys
    (1000, [0, 600, 901], [0, 600, 901], False),     # the second sequence ends inside a row group
    (1000, [0, 600, 901], [0, 500, 1000], True),     # both at once
])
def test_bsa_fwd_varlen_rows_without_keys(dev, length, cu_q, cu_k, far_rows):
    """Rows of a sequence whose kept blocks all lie past that sequence's keys
    (or whose sequence has no keys) are zero with lse -inf; a four-row group
    of the second-sequence kernel that straddles the sequence's end writes
    its rows past the end as zero. Against the fp32 varlen oracle."""
    from dfsattn_amd.workloads import DfsConfig, synth_qkv
    heads, d = 3, 128
    cfg = DfsConfig("t", (1, 1, length), heads, d, torch.bfloat16, seed=23)
    q, k, v = synth_qkv(cfg)
    nb = math.ceil(length / 128)
    g = torch.Generator().manual_seed(24)
    mask = torch.rand((heads, nb, nb), generator=g) < 0.4
    mask[:, torch.arange(nb), torch.arange(nb)] = True
    if far_rows:
        # rows 0..2 of every head keep only blocks 3.. (past 300 keys)
        mask[:, :3, :3] = False
        mask[:, :3, 5] = True
    layout = ScoringLayout(length, length, 16)
    ident = torch.arange(length, dtype=torch.int32)
    prep = ops.prepare_qkv(q.to(dev), k.to(dev), v.to(dev), ident.to(dev), layout, pool=False)
    row_ptr, col_idx = ops.mask_to_csr(mask.to(dev))
    out = torch.full((1, heads, length, d), 7.0, dtype=torch.float32, device=dev)
    cq = torch.tensor(cu_q, dtype=torch.int32, device=dev)
    ck = torch.tensor(cu_k, dtype=torch.int32, device=dev)
    _, lse = ops.bsa_fwd(prep, row_ptr, col_idx, out_dtype=torch.float32, out=out, cu_seqlens_q=cq,
                         cu_seqlens_k=ck, want_lse=True)
    got, lse = out.cpu(), lse.cpu()
    ref = orc.varlen_attention(q, k, v, mask, cu_q, cu_k)
    assert float((got - ref).abs().max()) <= 2e-2 and mean_rel(got, ref) <= 1e-3
    live = torch.zeros((heads, length), dtype=torch.bool)
    for (q0, q1), (k0, k1) in zip(zip(cu_q, cu_q[1:]), zip(cu_k, cu_k[1:])):
        nkb = math.ceil((k1 - k0) / 128)
        for r in range(q0, q1):
            live[:, r] = mask[:, (r - q0) // 128, :nkb].any(-1) if nkb > 0 else False
    assert bool((~live).any()), "the case must hold rows without keys"
    assert bool((got[0][~live] == 0).all())
    assert bool(torch.isneginf(lse[~live]).all())
    assert bool(torch.isfinite(lse[live]).all())


@pytest.mark.parametrize("case", ["bf16_d128", "f16_d64", "bf16_operands", "varlen", "q_beyond_f16"])
def test_bsa_fwd_q_source_matches_q_perm(dev, case):
    """dfs_bsa_fwd reading Q from the input through the permutation (q_src,
    q_rows; dfs_prepare_qkv then writes no q_perm) against the same call on
    the prepared q_perm and against fp32 masked attention: the two differ by
    the rounding of Q * scale * log2(e) to f16 only (one rounding from the
    input instead of two), and the second-sequence and scaled instances read
    the same source."""
    import math as _m
    from dfsattn_amd.workloads import DfsConfig, synth_qkv
    heads, d, length, dtype, pv = 3, 128, 1100, torch.bfloat16, torch.float16
    cu = None
    if case == "f16_d64":
        d, dtype = 64, torch.float16
    elif case == "bf16_operands":
        pv = torch.bfloat16
    elif case == "varlen":
        cu = [0, 900, length]
    cfg = DfsConfig("t", (1, 1, length), heads, d, torch.float32, seed=41)
    q, k, v = synth_qkv(cfg)
    if case == "q_beyond_f16":
        q[:, 1] *= 3e5  # head 1's Q exceeds the f16 range: the scaled instance, rows shifted in the kernel
    q, k, v = (x.to(dtype) for x in (q, k, v))
    perm = torch.randperm(length, generator=torch.Generator().manual_seed(42)).to(torch.int32)
    layout = ScoringLayout(length, length, 16)
    nb = _m.ceil(length / 128)
    mask = torch.rand((heads, nb, nb), generator=torch.Generator().manual_seed(43)) < 0.4
    mask[:, torch.arange(nb), torch.arange(nb)] = True
    row_ptr, col_idx = ops.mask_to_csr(mask.to(dev))
    kw = {}
    if cu is not None:
        cu_d = torch.tensor(cu, dtype=torch.int32, device=dev)
        kw = dict(cu_seqlens_q=cu_d, cu_seqlens_k=cu_d)
    outs = {}
    for q_operand in (True, False):
        prep = ops.prepare_qkv(q.to(dev), k.to(dev), v.to(dev), perm.to(dev), layout, operand_dtype=pv,
                               pool=False, q_operand=q_operand)
        assert (prep.q_perm is None) == (not q_operand)
        outs[q_operand] = ops.bsa_fwd(prep, row_ptr, col_idx, out_dtype=torch.float32, **kw).cpu()
    qp, kp, vp = (orc.apply_permutation(x.float(), perm.long()) for x in (q, k, v))
    ref = (orc.masked_attention(qp, kp, vp, mask) if cu is None else orc.varlen_attention(qp, kp, vp, mask, cu, cu))
    for q_operand, out in outs.items():
        ma, mr = float((out - ref).abs().max()), mean_rel(out, ref)
        tol = 1e-3 if pv == torch.float16 else 3e-3
        assert ma <= 2e-2 and mr <= tol, (q_operand, ma, mr)
    if pv == torch.bfloat16 or dtype == torch.float16:
        assert torch.equal(outs[True], outs[False])  # the same operand values either way
    elif case != "q_beyond_f16":  # (there one-hot rows may pick another key on a rounding)
        assert mean_rel(outs[False], outs[True]) < 5e-4
