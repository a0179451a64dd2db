"""Host-side logic and the C-ABI surface (CPU only: no kernel is launched)."""
import ctypes
import os
import re
import shutil
import subprocess

import numpy as np
import pytest
import torch

from dfsattn_amd import _lib, ops
from dfsattn_amd.layout import (ScoringLayout, TopkPolicy, csr_flops, block_flops, dense_policy,
                                hunyuan_policy, topk_count, wan_policy)
from oracle import dfs_oracle as orc

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "dfsattn_amd.h")


def test_library_exports_every_declared_symbol():
    text = open(HEADER).read()
    declared = set(re.findall(r"^\s*(?:int|int64_t|const char\*)\s+(dfs_\w+)\s*\(", text, flags=re.M))
    assert declared == set(_lib.SIGNATURES), declared ^ set(_lib.SIGNATURES)
    lib = _lib.lib()
    for name in declared:
        assert hasattr(lib, name), name
    assert lib.dfs_abi_version() == _lib.ABI_VERSION


@pytest.mark.parametrize("grid", [(4, 16, 16), (3, 5, 7), (1, 1, 1), (2, 3, 1), (21, 45, 80), (33, 45, 80)])
def test_hilbert_c_matches_numpy_oracle(grid):
    got = ops.hilbert3d_perm(*grid).numpy()
    assert np.array_equal(got, orc.hilbert3d_perm(*grid))


def test_abi_rejects_bad_arguments_without_launching():
    fake = ctypes.c_void_p(16)
    with pytest.raises(_lib.DfsKernelError, match="head_dim=96"):
        _lib.call("dfs_prepare_qkv", fake, fake, fake, fake, 2, 1000, 96, 0, 1000, 16, 16, 1,
                  fake, fake, fake, None, None, None, None, None, None)
    with pytest.raises(_lib.DfsKernelError, match="q_tile_size=24"):
        _lib.call("dfs_prepare_qkv", fake, fake, fake, fake, 2, 1000, 128, 0, 1000, 24, 16, 1,
                  fake, fake, fake, None, None, None, None, None, None)
    with pytest.raises(_lib.DfsKernelError, match="k_tile_size=48"):
        _lib.call("dfs_prepare_qkv", fake, fake, fake, fake, 2, 1000, 128, 0, 1000, 16, 48, 1,
                  fake, fake, fake, None, None, None, None, None, None)
    # scoring: tiles below 4 tokens, and the generic scorer without scores_out
    with pytest.raises(_lib.DfsKernelError, match="k_tile_size=2"):
        _lib.call("dfs_block_score_topk", fake, fake, fake, fake, 2, 128, 16, 2, 8, 8, 8, 8, 2, 8, 8,
                  fake, fake, None, None, None, 0, None)
    with pytest.raises(_lib.DfsKernelError, match="pass one"):
        _lib.call("dfs_block_score_topk", fake, fake, fake, fake, 2, 128, 8, 64, 8, 8, 8, 8, 2, 8, 8,
                  fake, fake, None, None, None, 0, None)
    with pytest.raises(_lib.DfsKernelError, match="k_pick"):
        _lib.call("dfs_topk_from_scores", fake, 2, 8, 8, 8, 8, 9, 8, 8, fake, fake, None, None)
    with pytest.raises(_lib.DfsKernelError, match="f16 inputs"):
        _lib.call("dfs_bsa_fwd", fake, fake, fake, fake, fake, 2, 1000, 128, 1, 0, 0.1, fake, 2,
                  None, None, None, None, 1, None, None, None, 0, None)
    with pytest.raises(_lib.DfsKernelError, match="n_seq=3"):
        _lib.call("dfs_bsa_fwd", fake, fake, fake, fake, fake, 2, 1000, 128, 1, 1, 0.1, fake, 2,
                  None, None, fake, fake, 3, None, None, None, 0, None)
    with pytest.raises(_lib.DfsKernelError, match="both cu_seqlens_q and cu_seqlens_k"):
        _lib.call("dfs_bsa_fwd", fake, fake, fake, fake, fake, 2, 1000, 128, 1, 1, 0.1, fake, 2,
                  None, None, fake, None, 2, None, None, None, 0, None)
    with pytest.raises(_lib.DfsKernelError, match="two sequences need cu_seqlens"):
        _lib.call("dfs_bsa_fwd", fake, fake, fake, fake, fake, 2, 1000, 128, 1, 1, 0.1, fake, 2,
                  None, None, None, None, 2, None, None, None, 0, None)
    with pytest.raises(_lib.DfsKernelError, match="q_src needs q_rows"):
        _lib.call("dfs_bsa_fwd", None, fake, fake, fake, fake, 2, 1000, 128, 1, 1, 0.1, fake, 2,
                  None, None, None, None, 1, None, fake, None, 0, None)
    with pytest.raises(_lib.DfsKernelError, match="bf16 Q/K operands need a bf16 q_src"):
        _lib.call("dfs_bsa_fwd", None, fake, fake, fake, fake, 2, 1000, 128, 0, 0, 0.1, fake, 2,
                  None, None, None, None, 1, None, fake, fake, 1, None)
    with pytest.raises(_lib.DfsKernelError, match="NULL operand"):
        _lib.call("dfs_bsa_fwd", None, fake, fake, fake, fake, 2, 1000, 128, 1, 1, 0.1, fake, 2,
                  None, None, None, None, 1, None, None, None, 0, None)
    with pytest.raises(_lib.DfsKernelError, match="head_dim=96"):
        _lib.call("dfs_prepare_fixup", fake, fake, fake, fake, 2, 1000, 96, fake, fake, fake, fake, fake, None)
    # the allocation-free scorer refuses block sums beyond its 96 MiB scratch
    # before touching a device (64 heads x 1000 x 1000 blocks = 256 MB)
    with pytest.raises(_lib.DfsKernelError, match="scratch holds 100663296"):
        _lib.call("dfs_block_score_topk_noalloc", fake, fake, fake, fake, 64, 128, 16, 16, 1000, 1000, 1000, 1000, 300,
                  1000, 1000, fake, fake, None, None)
    with pytest.raises(_lib.DfsKernelError, match="row_bytes"):
        _lib.call("dfs_permute_gather", fake, fake, fake, 1, 10, 10, 10, 3, None)
    with pytest.raises(_lib.DfsKernelError, match="positive"):
        _lib.call("dfs_hilbert3d_perm", 0, 4, 4, fake)


def test_ops_refuse_cpu_tensors():
    x = torch.zeros(1, 2, 128, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="ROCm GPU"):
        ops.permute_gather(x, torch.arange(128, dtype=torch.int32))


def test_config_shapes_and_policies():
    wan = ScoringLayout(75600, 75600, 16)
    assert (wan.q_blocks, wan.rows, wan.q_tiles, wan.k_tiles) == (591, 75648, 4728, 4728)
    pol = wan_policy(wan, 0.3)
    assert (pol.k_pick, pol.n_cand, pol.dense_row) == (177, 591, 591)
    assert pol.nnz(40) == 4184280
    assert pol.row_ptr(2)[-1] == 2 * 591 * 177
    hy = ScoringLayout(118800 + 256, 118800, 16)
    assert (hy.q_blocks, hy.video_blocks, hy.q_tiles, hy.k_tiles) == (931, 929, 7432, 7448)
    hp = hunyuan_policy(hy, 0.3)
    assert (hp.scored_rows, hp.n_cand, hp.k_pick, hp.dense_col, hp.dense_row) == (929, 928, 276, 928, 928)
    counts = hp.row_counts()
    assert (counts[:928] == 279).all() and (counts[928:] == 931).all()
    assert hp.nnz(24) == 6280920
    # schedule sparsities 0.3 / 0.2 / 0.1 -> Wan top-k 177 / 118 / 59 (0.2 * 591 = 118.2)
    assert [topk_count(s, 591) for s in (0.3, 0.2, 0.1)] == [177, 118, 59]
    d = dense_policy(wan)
    assert (d.row_counts() == 591).all()


def test_policy_errors_follow_the_reference():
    with pytest.raises(AssertionError):
        hunyuan_policy(ScoringLayout(118800 + 256, 118800, 16), 0.002)
    with pytest.raises(RuntimeError, match="tile view"):
        ScoringLayout(129 + 127, 129, 16)  # 2 video blocks + 127 text tokens > 2 blocks
    with pytest.raises(ValueError, match="block_size"):
        ScoringLayout(1000, 1000, 16, block=64)
    with pytest.raises(AssertionError, match="divisible"):
        ScoringLayout(1000, 1000, 48)
    with pytest.raises(RuntimeError, match="out of range"):
        wan_policy(ScoringLayout(1000, 1000, 16), 1.5)


def test_policy_row_counts_match_oracle_masks():
    for seq, video, ratio in ((1000, 1000, 0.3), (1060, 1000, 0.5), (1000, 1000, 0.05), (3256, 3000, 0.2)):
        lay = ScoringLayout(seq, video, 16)
        pol = wan_policy(lay, ratio) if seq == video else hunyuan_policy(lay, ratio)
        s = torch.rand(2, pol.scored_rows, pol.k_blocks)
        m = orc.mask_from_scores_wan(s, ratio) if seq == video else orc.mask_from_scores_hunyuan(s, ratio, seq, video)
        assert np.array_equal(m.sum(-1)[0].numpy(), pol.row_counts())


def test_flop_counts_use_valid_token_blocks():
    mask = np.ones((2, 3, 3), dtype=bool)
    assert block_flops(mask, 300, 64) == 4 * 64 * 300 * 300 * 2
    pol = wan_policy(ScoringLayout(300, 300, 16), 1.0)
    ptr = pol.row_ptr(2)
    cols = np.tile(np.arange(3), 6)
    assert csr_flops(ptr, cols, 2, 300, 64) == block_flops(mask, 300, 64)
    # cfg 1 nominal bound 35.10 TFLOP
    assert abs(4 * 128 * 128 * 128 * 4184280 / 1e12 - 35.10) < 0.01


def test_cu_seqlens_forms():
    """Host cu_seqlens: [0, L] and [0, L, L] are one sequence, [0, a, L] a
    split (including a = 0); other forms are refused. Device tensors are
    never read back (their checks run on the GPU tests)."""
    from dfsattn_amd.core import DfsCore
    check = DfsCore._host_split
    assert DfsCore._sequences(None, 300, torch.device("cpu"), "cu") is None
    assert check([0, 300], 300) is None
    assert check([0, 300, 300], 300) is None
    assert check([0, 250, 300], 300) == [0, 250, 300]
    assert check([0, 0, 300], 300) == [0, 0, 300]
    for bad in ([0, 100, 200, 300], [1, 300], [0, 310, 300], [0, 200], [0, 200, 100, 300]):
        with pytest.raises(NotImplementedError):
            check(bad, 300)


@pytest.mark.parametrize("grid", [(1, 4, 4), (3, 5, 7), (2, 8, 8), (5, 3, 9), (1, 1, 1), (4, 16, 16), (2, 45, 80)])
def test_token_orders_match_oracle(grid):
    from dfsattn_amd.utils import order as od
    f, h, w = grid
    cases = {
        "hilbert2d": (od.hilbert2d_perm(f, h, w), orc.hilbert2d_perm(f, h, w)),
        "morton3d": (od.morton3d_perm(f, h, w), orc.morton_perm(f, h, w, per_frame=False)),
        "morton2d": (od.morton2d_perm(f, h, w), orc.morton_perm(f, h, w, per_frame=True)),
        "hwf": (od.hwf(f, h, w), orc.axis_order_perm(f, h, w, "hwf")),
        "fwh": (od.fwh(f, h, w), orc.axis_order_perm(f, h, w, "fwh")),
        "blk": (od.block3d_perm(f, h, w, 4, 4, 4), orc.block3d_perm(f, h, w, 4, 4, 4)),
        "blk_ragged": (od.block3d_perm(f, h, w, 2, 3, 5), orc.block3d_perm(f, h, w, 2, 3, 5)),
    }
    for name, (got, ref) in cases.items():
        assert got.dtype == torch.long and np.array_equal(got.numpy(), ref), name


def test_morton_bit_spreading_and_dispatch():
    from dfsattn_amd.utils import order as od
    v = torch.tensor([0, 1, 2, 3, 7, (1 << 20), (1 << 21) + 5])
    assert od.part1by2_tensor(v).tolist() == [0, 1, 8, 9, 0b1001001, 1 << 60, 0b1000001]
    assert od.part1by1_tensor(torch.tensor([1, 2, 3, (1 << 31), (1 << 32) + 1])).tolist() == [1, 4, 5, 1 << 62, 1]
    assert od.morton3D_tensor(torch.tensor([1, 0, 0]), torch.tensor([0, 1, 0]), torch.tensor([0, 0, 1])).tolist() == [1, 2, 4]
    assert od.video_perm_for("org", 2, 3, 4) is None
    for name in od.ORDERS[1:]:
        p = od.video_perm_for(name, 3, 8, 8)
        assert sorted(p.tolist()) == list(range(192)), name
    assert torch.equal(od.video_perm_for("blk", 3, 8, 8), od.block3d_perm(3, 8, 8, 4, 4, 4))
    with pytest.raises(ValueError):
        od.video_perm_for("zigzag", 1, 2, 2)


def test_workspace_size_by_tile_pair():
    """The one-pass workspace exists for equal 16- or 32-token tiles only;
    other valid pairs report 0 (two-pass generic scorer), invalid ones -1."""
    ws = _lib.lib().dfs_block_score_topk_workspace_size
    assert ws(40, 16, 16, 591, 591) > 0 and ws(40, 32, 32, 591, 591) > 0
    for qt, kt in ((8, 64), (16, 32), (128, 4), (64, 64), (8, 8)):
        assert ws(40, qt, kt, 591, 591) == 0
    for qt, kt in ((2, 16), (16, 24), (256, 16), (0, 16)):
        assert ws(40, qt, kt, 591, 591) == -1


def test_noalloc_wrapper_runs_under_the_tensors_device(monkeypatch):
    """ops.block_score_topk_noalloc makes the tensors' device current around
    the C call (the library takes its scratch from the stream's device, and
    the launch and the stream then agree whichever device the caller has
    current). Host logic only: the device context and the C call are
    recorded, nothing runs on a GPU."""
    from types import SimpleNamespace
    from dfsattn_amd.layout import ScoringLayout, wan_policy

    events = []

    class FakeDeviceCtx:
        def __init__(self, dev):
            self.dev = dev

        def __enter__(self):
            events.append(("enter", self.dev))

        def __exit__(self, *exc):
            events.append(("exit", self.dev))

    target = torch.device("cuda", 3)
    fake_t = SimpleNamespace(device=target)
    layout = ScoringLayout(1024, 1024, 16)
    pol = wan_policy(layout, 0.3)
    prep = SimpleNamespace(q_hi=fake_t, q_lo=fake_t, k_hi=fake_t, k_lo=fake_t, q_perm=None, k_perm=fake_t,
                           device=target, heads=2, head_dim=64, layout=layout)
    real_empty = torch.empty
    monkeypatch.setattr(ops, "_require_device", lambda *a: None)
    monkeypatch.setattr(ops, "_require_int32", lambda **k: None)
    monkeypatch.setattr(ops, "_ptr", lambda t: None)
    monkeypatch.setattr(ops, "_stream", lambda t: None)
    monkeypatch.setattr(ops.torch, "empty", lambda *a, device=None, **k: real_empty(*a, **k))
    monkeypatch.setattr(ops.torch.cuda, "device", FakeDeviceCtx)
    monkeypatch.setattr(ops._lib, "call", lambda name, *args: events.append(("call", name, args[6], args[7])))
    row_ptr = torch.from_numpy(pol.row_ptr(2))
    ops.block_score_topk_noalloc(prep, pol, row_ptr)
    assert events == [("enter", target), ("call", "dfs_block_score_topk_noalloc", 16, 16), ("exit", target)]


@pytest.mark.parametrize("heads,length,text,kept", [
    (1, 100, 0, 1), (1, 7872, 0, 62), (2, 1024, 0, 2), (9, 9000, 0, 20), (40, 75600, 0, 177), (24, 119056, 256, 279),
    (2, 30250, 250, 60), (8, 6200, 200, 14), (16, 5000, 0, 12), (3, 200, 100, 0), (1, 5, 4, 1)])
def test_attention_plan_covers_every_block_once(heads, length, text, kept):
    """The workgroup -> (head, query block, part) map of dfs_bsa_fwd_parts,
    restated here, visits every part of every query block exactly once under
    the plan, partial slots are distinct and lie inside the workspace, and
    the combining kernel's map finds the same blocks."""
    from dfsattn_amd.layout import attention_plan, head_chunks
    Qb = -(-length // 128)
    c = head_chunks(heads, Qb * 128, 128)
    assert c in (1, 2, 4, 8) and heads * c % 8 == 0
    long_row = (length - text) // 128 if text else Qb
    lp, full, parts = attention_plan(heads, Qb, long_row, kept, Qb, c)
    assert 1 <= lp <= 64 and 1 <= parts <= 64 and 0 <= full <= -(-heads * c // 8) * -(-long_row // c)
    S, n_long = -(-long_row // c), Qb - long_row
    long_x = -(-heads * n_long // 8)
    in_order = -(-heads * c // 8) * S  # ordinary blocks per XCD
    full_k = full if parts > 1 else in_order
    split_long = 8 * long_x if lp > 1 else 0
    split_tail = 8 * (in_order - full_k) if parts > 1 else 0
    size = _lib.lib().dfs_bsa_fwd_workspace_size(heads, length, 128, long_row, lp, full, parts, c)
    slots = split_long * lp + split_tail * parts
    assert size == slots * 128 * 130 * 4
    per = long_x * lp + full_k + (in_order - full_k) * parts
    seen, used = {}, {}

    def ordinary(x, i):
        g = (i // S) * 8 + x
        h = g // c
        qb = ((g + h) & (c - 1)) * S + i % S
        return (h, qb) if h < heads and qb < long_row else None

    for b in range(8 * per):
        x, j = b & 7, b >> 3
        if j < long_x * lp:
            g = (j // lp) * 8 + x
            blk = (g // n_long, long_row + g % n_long) if g < heads * n_long else None
            piece, pieces, slot = j % lp, lp, g * lp + j % lp
        else:
            j -= long_x * lp
            if parts > 1 and j >= full_k:
                t, piece = divmod(j - full_k, parts)
                blk, pieces = ordinary(x, full_k + t), parts
                slot = split_long * lp + (t * 8 + x) * parts + piece
            else:
                blk, piece, pieces, slot = ordinary(x, j), 0, 1, None
        if blk is None:
            continue
        seen.setdefault(blk, []).append((piece, pieces))
        if pieces > 1:
            assert 0 <= slot < slots and slot not in used
            used[slot] = (blk, piece)
    assert set(seen) == {(h, qb) for h in range(heads) for qb in range(Qb)}
    for got in seen.values():
        assert sorted(got) == [(i, got[0][1]) for i in range(got[0][1])]
    for r in range(split_long + split_tail):  # the combining kernel's blocks
        if r < split_long:
            blk = (r // n_long, long_row + r % n_long) if r < heads * n_long else None
            base, n = r * lp, lp
        else:
            t = r - split_long
            blk, base, n = ordinary(t & 7, full_k + (t >> 3)), split_long * lp + t * parts, parts
        if blk is not None:
            assert [used[base + i] for i in range(n)] == [(blk, i) for i in range(n)]


def test_call_checks_its_arguments_without_launching():
    """dfs_call refuses sizes, phases and workspaces it cannot run before it
    touches a device."""
    from dfsattn_amd.ops import _call_template
    layout = ScoringLayout(1000, 1000, 16)
    template, size, nnz = _call_template(layout, wan_policy(layout, 0.3), 2, 128, torch.bfloat16, torch.float16, True)
    assert nnz == wan_policy(layout, 0.3).nnz(2) and size > 2 * 2 * 1024 * 128 * 2
    ref = lambda a: ctypes.byref(a)  # noqa: E731

    def args(**kw):
        a = _lib.CallArgs.from_buffer_copy(template)
        a.q = a.k = a.v = a.perm = a.row_ptr = a.col_idx = a.out = a.workspace = 256
        for name, value in kw.items():
            setattr(a, name, value)
        return a

    for bad, text in ((dict(workspace_bytes=size - 1), "workspace"), (dict(workspace=None), "workspace"),
                      (dict(workspace=264), "workspace"), (dict(head_dim=96), "head_dim=96"),
                      (dict(q_tile=24), "q_tile=24"), (dict(video_len=1001), "video_len=1001"),
                      (dict(k_blocks=9), "policy"), (dict(parts=0), "parts=0"), (dict(long_row=9), "long_row=9")):
        with pytest.raises(_lib.DfsKernelError, match=text):
            _lib.call("dfs_call", ref(args(**bad)), 7, None)
    with pytest.raises(_lib.DfsKernelError, match="phases=8"):
        _lib.call("dfs_call", ref(args()), 8, None)
    with pytest.raises(_lib.DfsKernelError, match="NULL"):
        _lib.call("dfs_call", None, 7, None)
    assert _lib.lib().dfs_call_workspace_size(ref(args(head_dim=96))) == -1


HEAD_RANGE_MODEL = r"""
#include <cstdio>
#include "head_range.h"
struct P { const int32_t* exps; int32_t* q_marks; int H, scale_all; };
int main() {
  // exponent words of one head: Q's, K's; marked: another workgroup finds Q beyond the range
  for (int marks = 0; marks < 2; ++marks)
    for (int q = 0; q < 2 - marks; ++q)
      for (int k = 0; k < 2; ++k)
        for (int all = 0; all < 2; ++all) {
          int32_t exps[3] = {q, k, 0};
          const P p{exps, marks ? exps : nullptr, 1, all};
          const bool first = dfs::common_skips(p, 0);   // the workgroup's first wave asks
          if (marks) p.q_marks[0] = 1;                  // a workgroup of the same launch marks the head
          const bool last = dfs::common_skips(p, 0);    // its last wave asks
          printf("%d %d %d %d %d %d %d\n", marks, q, k, all, first, last, dfs::head_scaled(p, 0));
        }
}
"""


def _run_on_host(tmp_path, source):
    """Output lines, as integers, of a program over the kernels' host code."""
    src, exe = tmp_path / "model.cpp", tmp_path / "model"
    src.write_text(source)
    csrc = os.path.join(os.path.dirname(_lib.__file__), "csrc")
    subprocess.run(["g++", "-std=c++17", "-I", csrc, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    return [[int(x) for x in line.split()] for line in out.splitlines()]


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_common_instance_exit_does_not_depend_on_marks_of_its_launch(tmp_path):
    """The waves of a workgroup decide one by one whether the scaled instance
    has their head, so the answer may not change while the common instance
    runs and marks heads; the launches behind it see the mark. The rule of
    csrc/head_range.h, compiled for the host."""
    lines = _run_on_host(tmp_path, HEAD_RANGE_MODEL)
    assert len(lines) == 12
    for marks, q, k, scale_all, first, last, behind in lines:
        assert first == last == (scale_all or q or k)
        assert behind == (scale_all or q or k or marks)


SCALED_BLOCK_MODEL = r"""
#include <cstdio>
#include "head_range.h"
struct P { const int32_t* exps; int32_t *q_marks, *q_block_marks; int H, Qb, scale_all; };
int main() {
  for (int marks = 0; marks < 2; ++marks)
    for (int k = 0; k < 2; ++k)
      for (int all = 0; all < 2; ++all) {
        int32_t exps[6] = {0, 1, 0, k, 0, 0}, blocks[6] = {1, 0, 0, 0, 1, 0};  // of head 1, block 1 is marked
        const P p{exps, marks ? exps : nullptr, marks ? blocks : nullptr, 2, 3, all};
        printf("%d %d %d %d %d %d %d\n", marks, k, all, dfs::head_scaled(p, 1), dfs::scaled_block(p, 1, 0),
               dfs::scaled_block(p, 1, 1), dfs::scaled_block(p, 1, 2));
      }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_scaled_instance_redoes_marked_blocks_only(tmp_path):
    """Of a head whose Q alone left the range, found by the common instance,
    the scaled instance does the marked query blocks; of any other head it has,
    all."""
    lines = _run_on_host(tmp_path, SCALED_BLOCK_MODEL)
    assert len(lines) == 8
    for marks, k, scale_all, takes, *blocks in lines:
        assert takes
        assert blocks == ([0, 1, 0] if marks and not k and not scale_all else [1, 1, 1])


@pytest.mark.parametrize("shape,how", [
    ((1, 2, 40, 64), "contiguous"), ((3, 40, 64), "contiguous"),  # contiguous, off 16 bytes
    ((1, 1, 40, 64), "one head"), ((1, 2, 1, 64), "one row"),     # any stride on an axis of one
    ((1, 2, 40, 64), "rows"), ((1, 2, 40, 64), "token"), ((1, 2, 40, 64), "channels")])
@pytest.mark.parametrize("offset", [0, 1, 8])
def test_rows_in_place_gives_16_byte_rows(shape, how, offset):
    """What the call passes to the kernels: the same rows, on 16-byte
    boundaries and strides, whatever the caller's offset and strides."""
    n = 1
    for s in shape:
        n *= s
    buf = torch.arange(4 * n + offset + 64, dtype=torch.float32).to(torch.float16)[offset:]
    h, l, d = shape[-3:]
    strides = {"contiguous": (l * d, d, 1), "one head": (3, d, 1), "one row": (d, 5, 1), "rows": (l * (d + 3), d + 3, 1),
               "token": (d, h * d, 1), "channels": (2 * l * d, 2 * d, 2)}[how]
    x = buf.as_strided(shape, ((7,) if len(shape) == 4 else ()) + strides)
    x.copy_(torch.randn(shape))
    y, sh, sl = ops._rows_in_place(x)
    assert y.data_ptr() % 16 == 0 and sh % 8 == 0 and sl % 8 == 0
    room = y.untyped_storage().nbytes() // 2 - y.storage_offset()
    assert (h - 1) * sh + (l - 1) * sl + d <= room
    assert torch.equal(y.as_strided((h, l, d), (sh, sl, 1)), x.reshape(h, l, d))
    if x.data_ptr() % 16 == 0 and how in ("contiguous", "token", "one head", "one row"):
        assert y.data_ptr() == x.data_ptr()  # read where it is


def test_cached_layouts_and_policies_hold_plain_integers():
    """Sizes that compare equal share a cache entry: one call's numpy, tensor
    or refused float sizes leave nothing of their type to the next call."""
    from dfsattn_amd.layout import scoring_layout
    plain = (1511, 1401, 16, 128, 32)
    for sizes in ((1511, np.int64(1401), 16, 128, 32), (1511, torch.tensor(1401), np.int32(16), 128, torch.tensor(32)),
                  (1511, 1401, 16, 128, 32)):
        lay = scoring_layout(*sizes)
        assert lay == ScoringLayout(*plain[:4], k_tile=32)
        assert all(type(x) is int for x in (lay.seq_len, lay.video_len, lay.tile, lay.block, lay.k_tile))
    for i in range(1, 5):  # refused, as they always were further on, before and after the plain sizes are known
        for base in ((1611, 1401, 16, 128, 32), plain):
            sizes = [float(x) if j == i else x for j, x in enumerate(base)]
            with pytest.raises(TypeError):
                scoring_layout(*sizes)
            assert type(scoring_layout(*base).video_len) is int
    with pytest.raises(AssertionError, match="q_tile_size"):
        scoring_layout(1511, 1401, 15.5, 128, 32)
    assert scoring_layout(1511, 1401, 16, 128, None).k_tile == 16
    hunyuan_policy(ScoringLayout(1521, 1401.0, 16), 0.5)
    pol = hunyuan_policy(ScoringLayout(1521, 1401, 16), 0.5)
    assert all(type(x) is int for x in (pol.n_cand, pol.k_pick, pol.dense_col, pol.dense_row))
