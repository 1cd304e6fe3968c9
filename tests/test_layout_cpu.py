"""How the binding reads a 2-D view's layout (dot.py `_layout`, `aligned_rows`,
`plan_for`), on CPU tensors: row-major, a transposed view of row-major storage
(K-major B), and the stride of a size-1 dimension, which says nothing about
the layout.  Planning runs on the host; nothing here launches."""
import importlib

import pytest

import triton_ext_amd as tx

txdot = importlib.import_module("triton_ext_amd.dot")  # the module (the package exports dot())


def _t(shape, dtype_name="bfloat16"):
    import torch
    return torch.zeros(shape, dtype=getattr(torch, dtype_name))


def test_layout_kinds():
    import torch
    st = _t((220, 8))                     # [N][K'] storage, rows 16 bytes apart
    assert txdot._layout(st[:, :5]) == ("row", 8)
    assert txdot._layout(st[:, :5].t()) == ("col", 8)       # K-major B, K = 5
    assert txdot._layout(st[:, :1].t()) == ("col", 8)       # K = 1: one row, elements 8 apart
    assert txdot._layout(_t((1, 300)).t()) == ("col", 300)  # N = 1, adjacent elements: K-major
    assert txdot._layout(_t((1, 300)).t(), col_ok=False) == ("row", 1)  # or one row-major column
    assert txdot._layout(st[:, :5].t(), col_ok=False)[0] is None
    assert txdot._layout(_t((64, 64))[::2, ::2])[0] is None  # neither rows nor columns contiguous
    assert txdot._layout(torch.zeros(1, 1)) == ("row", 1)


def test_plan_k1_kmajor_b():
    """q @ k.T with one head dim: B = k.t() is [1, N] with elements ldk apart."""
    a = txdot.aligned_rows(_t((5, 8))[:, :1])
    b = _t((220, 8))[:, :1].t()
    assert txdot.aligned_rows(b) is b     # already 16-byte columns
    p = txdot.plan_for(a, b, tx.F32)
    assert p.desc.flags & tx.FLAG_B_KMAJOR and p.desc.ldb == 8 and p.desc.K == 1


@pytest.mark.parametrize("dtype_name,txt", [("int8", tx.I32), ("bfloat16", tx.F32)])
def test_plan_single_column_b(dtype_name, txt):
    """N = 1, B = x.t() for x [1, K]: row-major (any dtype), after the copy into
    16-byte rows that its 1-element pitch needs."""
    K = 300
    a = txdot.aligned_rows(_t((40, K), dtype_name))
    b = txdot.aligned_rows(_t((1, K), dtype_name).t(), col_ok=False)
    assert b.shape == (K, 1) and (b.stride(0) * b.element_size()) % 16 == 0
    p = txdot.plan_for(a, b, txt, ldc=4)  # C rows of one 4-byte element, 16 bytes apart
    assert not p.desc.flags & tx.FLAG_B_KMAJOR and p.desc.N == 1


def test_plan_8bit_transposed_b():
    """An int8 B given as a transposed view (a weight kept [N][K]) runs K-major, unscaled
    (int32 C) or W8A8; with a block that has no K-major form it is copied row-major."""
    bt = _t((64, 304), "int8")[:, :300].t()      # [300][64] view, columns 304 bytes apart
    a = txdot.aligned_rows(_t((16, 300), "int8"), col_ok=False)
    for c, sm in ((tx.I32, tx.SCALE_NONE), (tx.BF16, tx.SCALE_ROWCOL)):
        assert txdot._b_kmajor_ok(a, bt, c, sm, (0, 0, 0), 0)
        assert txdot.aligned_rows(bt, col_ok=True) is bt
        p = txdot.plan_for(a, bt, c, sm)
        assert p.desc.flags & tx.FLAG_B_KMAJOR and p.desc.ldb == 304
    assert not txdot._b_kmajor_ok(a, bt, tx.BF16, tx.SCALE_ROWCOL, (256, 224, 128), 0)
    b = txdot.aligned_rows(bt, col_ok=False)
    assert b.stride(1) == 1 and b.shape == (300, 64)
    p = txdot.plan_for(a, b, tx.BF16, tx.SCALE_ROWCOL, block=(256, 224, 128))
    assert not p.desc.flags & tx.FLAG_B_KMAJOR


@pytest.mark.parametrize("dtype_name,txt,M,tile,other", [
    ("int8", tx.I32, 16, (16, 128, 128), (256, 224, 128)),
    ("int8", tx.I32, 600, (256, 256, 128), (256, 224, 128)),
    ("bfloat16", tx.F32, 16, (16, 64, 128), (128, 128, 64)),
    ("bfloat16", tx.F32, 100, (256, 256, 64), (64, 64, 32))])
def test_transposed_b_with_an_explicit_block(dtype_name, txt, M, tile, other):
    """K-major B where the tile has that form: the planner's own choice, or that tile asked
    for by name; another block copies B row-major (dot) or is refused (plan_for)."""
    bt = _t((64, 304), dtype_name)[:, :300].t()
    a = txdot.aligned_rows(_t((M, 300), dtype_name), col_ok=False)
    for blk in ((0, 0, 0), tile):
        assert txdot._b_kmajor_ok(a, bt, txt, tx.SCALE_NONE, blk, 0)
        p = txdot.plan_for(a, bt, txt, block=blk)
        assert p.desc.flags & tx.FLAG_B_KMAJOR and (p.desc.block_m, p.desc.block_n,
                                                    p.desc.block_k) == tile
    assert not txdot._b_kmajor_ok(a, bt, txt, tx.SCALE_NONE, other, 0)
    b = txdot.aligned_rows(bt, col_ok=False)
    assert b.stride(1) == 1
    assert not txdot.plan_for(a, b, txt, block=other).desc.flags & tx.FLAG_B_KMAJOR
    with pytest.raises(ValueError, match="transposed view"):
        txdot.plan_for(a, bt, txt, block=other)


def test_plan_rejects_a_transposed_a():
    a = _t((64, 64)).t()[:, :32]          # columns contiguous: A must be row-major
    with pytest.raises(ValueError):
        txdot.plan_for(a, _t((32, 16)), tx.F32)


def _overlapping(kind):
    """Views of fewer elements than they show: 16 bytes apart or 0, on an aligned base."""
    import torch
    r = torch.arange(4096, dtype=torch.float32).to(torch.bfloat16)
    return {"row": r[:320].expand(64, 320),                  # every row the same: stride 0
            "col": r[:64, None].expand(64, 320),             # every column the same (rows of one value)
            "kmajor": r[:64].expand(320, 64).t(),            # the same as a transposed view
            "column": r[:1, None].expand(64, 1),
            "window": r.unfold(0, 320, 8)[:64]}[kind]        # rows that share elements


@pytest.mark.parametrize("kind", ["row", "col", "kmajor", "column", "window"])
@pytest.mark.parametrize("col_ok", [False, True])
def test_overlapping_rows_are_copied(kind, col_ok):
    """A stride of 0 reads as "packed" in a descriptor: such a view, and rows that overlap, are
    copied to storage of their own, and a plan of the view itself is refused."""
    import torch
    t = _overlapping(kind)
    c = txdot.aligned_rows(t, col_ok=col_ok)
    assert c is not t and torch.equal(c, t)
    lies, ld = txdot._layout(c, col_ok)
    n, length = c.shape if lies == "row" else c.shape[::-1]
    assert ld >= length and ld % 8 == 0 and c.untyped_storage().nbytes() >= ((n - 1) * ld + length) * 2
    other, ldc = _t((16, 64)), -(-t.shape[1] // 8) * 8
    with pytest.raises(ValueError):
        txdot.plan_for(other, t, tx.BF16, ldc=ldc)
    assert txdot.plan_for(other, txdot.aligned_rows(t), tx.BF16, ldc=ldc).desc.K == 64
    if kind in ("row", "window"):
        with pytest.raises(ValueError):
            txdot.plan_for(t, _t((320, 64)), tx.BF16)
        a = txdot.aligned_rows(t, col_ok=False)
        assert txdot.plan_for(a, _t((320, 64)), tx.BF16).desc.lda >= 320


def test_single_rows_of_any_stride_are_not_copied():
    import torch
    t = torch.as_strided(_t((64,)), (1, 64), (0, 1))  # one row: its stride says nothing
    assert txdot.aligned_rows(t, col_ok=False) is t
    assert txdot.plan_for(t, _t((64, 64)), tx.BF16).desc.lda == 64


@pytest.mark.parametrize("dtype_name", ["bfloat16", "float8_e5m2"])
def test_attention_broadcast_heads_are_copied(dtype_name, monkeypatch):
    """k and v of one head shown to all (a stride of 0) reach the plan as packed copies; a
    dimension of size 1 may have any stride."""
    import torch
    seen = {}

    class Planned(Exception):
        pass

    def plan(*args, strides=None, **kw):
        seen.update(strides)
        raise Planned

    monkeypatch.setattr(txdot.capi, "attn_plan", plan)
    q = _t((1, 4, 128, 32), dtype_name)
    k = _t((1, 1, 128, 32), dtype_name).expand(1, 4, 128, 32)
    v = _t((1, 1, 32, 128), dtype_name).expand(1, 4, 32, 128).permute(0, 1, 3, 2) \
        if dtype_name == "float8_e5m2" else k
    with pytest.raises(Planned):
        txdot.attention(q, k, v, False, 0.5)
    rows = 128 if dtype_name == "float8_e5m2" else 32
    assert seen["k"][1:] == (128 * 32, 32) and seen["v"][1:] == (128 * 32, rows)


def test_broadcast_out_is_refused():
    import torch
    with pytest.raises(ValueError, match="16 bytes apart"):
        txdot._out_ldc(torch.zeros(1, 64).expand(16, 64))
    assert txdot._out_ldc(torch.zeros(16, 64)) == 64
