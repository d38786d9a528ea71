"""The attention kernels' routes against each other, bit for bit: long decode rows, batched decode rows and prompt rows run
different kernels whose partials are the same chains (the prompt and short decode routes are compared with the oracle in
test_gpu_model.py)."""
import struct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gw():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import gwenedeg_amd
    return gwenedeg_amd


def _bits_equal(a, b):
    return np.array_equal(np.ascontiguousarray(a, np.float32).view(np.uint32), np.ascontiguousarray(b, np.float32).view(np.uint32))


# decode rows go to k_attn_decode4 once heads x key blocks exceed the CUs (256): 8 heads (4 vectors per KV head, head_dim
# 128) from 32 blocks, 8 heads on one KV head (two groups of vectors, 64) likewise, 16 heads on one (four) from 16, 8
# KV heads of one vector (32); the row's position at the first and last places of a block, of a wave's 64 positions, of a
# tile and inside them
@pytest.mark.parametrize("kvt", ["f16", "bf16"])
@pytest.mark.parametrize("shape,base", [("tiny_gqa4", 8192), ("tiny_hd64", 8192), ("tiny_kv16", 4096), ("tiny_hd32", 8192)])
def test_long_decode_equals_the_other_routes(gw, synth_models, shape, base, kvt):
    m = gw.Model(synth_models(shape), ctx_len=9216)
    t = gw.RQ_KV_F16 if kvt == "f16" else gw.RQ_KV_BF16
    c, cb = m.ctx(max_batch=1), m.ctx(max_batch=8)
    a, b = m.seq(9216, t), m.seq(9216, t)
    a.fill_synthetic(base + 256, 77)
    b.fill_synthetic(base + 256, 78)
    for off in (0, 1, 13, 15, 62, 63, 64, 130, 254, 255):
        n = base + off
        a.truncate(n)
        one = [c.decode(a, 5), c.decode(a, 9)]
        a.truncate(n)
        rows = cb.prefill(a, np.array([5, 9], np.int32), mode=gw.RQ_LOGITS_ALL)
        a.truncate(n)
        b.truncate(n)
        batch = cb.forward_batch([gw.Segment(a, [5]), gw.Segment(b, [7])])[0]
        assert _bits_equal(one[0], rows[0]) and _bits_equal(one[1], rows[1]), f"position {n}: decode against a prompt's rows"
        assert _bits_equal(one[0], batch[0]), f"position {n}: decode against a batch"
        a.truncate(n)
        a.fill_synthetic(base + 256, 77)
        b.fill_synthetic(base + 256, 78)


def _first_tensor(path):
    """Byte offset of a GGUF file's tensor data (its first tensor is the embedding table, Q8_0 rows)."""
    raw = open(path, "rb").read(1 << 20)
    at = 24

    def u(n):
        nonlocal at
        at += n
        return int.from_bytes(raw[at - n:at], "little")

    def text():
        nonlocal at
        n = u(8)
        at += n
        return raw[at - n:at].decode()

    size = {0: 1, 1: 1, 2: 2, 3: 2, 4: 4, 5: 4, 6: 4, 7: 1, 10: 8, 11: 8, 12: 8}
    tensors, metas = struct.unpack_from("<QQ", raw, 8)
    for _ in range(metas):
        text()
        t = u(4)
        if t == 8:
            text()
        elif t == 9:
            et, n = u(4), u(8)
            for _ in range(n):
                if et == 8:
                    text()
                else:
                    at += size[et]
        else:
            at += size[t]
    for i in range(tensors):
        name, dims = text(), [u(8) for _ in range(u(4))]
        u(4)
        off = u(8)
        if i == 0:
            assert name == "token_embd.weight" and off == 0 and len(dims) == 2
    return (at + 31) // 32 * 32


# a row that is not finite (a NaN in its token's embedding) stays out of the rows before it: in the row block's MFMAs its
# V meets their zero weights
@pytest.mark.parametrize("shape,n,bad", [("tiny_gqa4", 40, 17), ("tiny_gqa4", 40, 2), ("tiny_hd64", 300, 261)])
def test_a_later_nan_row_changes_no_earlier_row(gw, tmp_path, shape, n, bad):
    from gwenedeg_amd import synth
    path = synth.write_gguf(str(tmp_path / "m.gguf"), shape, seed=5)
    at = _first_tensor(path)
    nan_token, dim = 11, synth.SHAPES[shape]["dim"]
    with open(path, "r+b") as f:
        f.seek(at + nan_token * (dim // 32) * 34)
        f.write(struct.pack("<H", 0x7e00))
    m = gw.Model(path, ctx_len=512)
    c = m.ctx(max_batch=512)
    ids = np.random.default_rng(3).integers(20, 900, n).astype(np.int32)
    clean = c.prefill(m.seq(512), ids, mode=gw.RQ_LOGITS_ALL)
    ids[bad] = nan_token
    got = c.prefill(m.seq(512), ids, mode=gw.RQ_LOGITS_ALL)
    assert _bits_equal(got[:bad], clean[:bad])
    assert np.isnan(got[bad]).all() and np.isnan(got[n - 1]).all()
