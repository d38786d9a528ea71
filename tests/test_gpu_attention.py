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
    _routes_agree(gw, synth_models(shape), base, kvt)


# groups of vectors that are not four: 2 and 3 vectors per KV head, 6 (a group of four, then two), 7 (four, then three) and, for
# head_dim 32, 5 (four, then one); k_attn_decode4 from 22, 19 and 7 key blocks
@pytest.mark.parametrize("kvt", ["f16", "bf16"])
@pytest.mark.parametrize("heads,kv,hd,base", [(12, 6, 128, 6144), (12, 4, 64, 6144), (12, 2, 128, 6144), (14, 2, 128, 5120),
                                              (40, 8, 32, 4096)])
def test_long_decode_of_uneven_groups(gw, tmp_path, heads, kv, hd, base, kvt):
    from gwenedeg_amd import synth
    path = synth.write_gguf(str(tmp_path / "m.gguf"), "tiny_gqa4", seed=6, n_heads=heads, n_kv_heads=kv, head_dim=hd)
    _routes_agree(gw, path, base, kvt)


def _routes_agree(gw, path, base, kvt):
    m = gw.Model(path, ctx_len=9216)
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
@pytest.mark.parametrize("kvt", ["f16", "bf16"])
@pytest.mark.parametrize("shape,n,bad", [("tiny_gqa4", 40, 17), ("tiny_gqa4", 40, 2), ("tiny_hd64", 300, 261), ("tiny_hd32", 270, 13)])
def test_a_later_nan_row_changes_no_earlier_row(gw, tmp_path, shape, n, bad, kvt):
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
    t = gw.RQ_KV_F16 if kvt == "f16" else gw.RQ_KV_BF16
    clean = c.prefill(m.seq(512, t), ids, mode=gw.RQ_LOGITS_ALL)
    ids[bad] = nan_token
    got = c.prefill(m.seq(512, t), ids, mode=gw.RQ_LOGITS_ALL)
    assert _bits_equal(got[:bad], clean[:bad])
    assert np.isnan(got[bad]).all() and np.isnan(got[n - 1]).all()


def _tiles(x, bf, v):
    """[blocks, 256, kv heads, hd] 16-bit values in a layer's cache order (blocks, heads, tiles of 16 positions)."""
    nb, _, nkv, hd = x.shape
    x = x.reshape(nb, 16, 16, nkv, hd).transpose(0, 3, 1, 2, 4)  # block, head, tile, position, dim
    if v:
        return np.ascontiguousarray(x.reshape(*x.shape[:4], hd // 32, 2, 16).swapaxes(-1, -2) if bf else x).reshape(-1)
    x = x.swapaxes(-1, -2)
    return np.ascontiguousarray(x.reshape(*x.shape[:3], hd // 2, 2, 16).swapaxes(-1, -2) if bf else x).reshape(-1)


# Sums around the smallest normal float, where flushed denormals decide the bits: each block's weights are e^-82 .. 4.5e-38 (the
# exponential's clamp) but for its position 7, whose V is zero; V from 1 down to the cache type's subnormals (bf16: products,
# sums and V itself are denormal), half of it zero. The four kernels of the fp32 chains (VALU: k_attn_decode; matrix cores:
# k_attn_decode4, k_attn_part4, k_attn_part) against the oracle with this CPU's flush modes on; the cache behind the row is NaN
@pytest.mark.parametrize("kvt", ["f16", "bf16"])
@pytest.mark.parametrize("hd,pos", [(128, 611), (64, 512 + 255), (128, 32 * 256 + 100), (64, 32 * 256 + 15)])
def test_denormals_are_flushed_alike(gw, synth_models, hd, pos, kvt):
    import ctypes

    import torch
    from oracle import oracle as orc
    gw.Model(synth_models("tiny"), ctx_len=64)  # (the device's tables)
    P, I, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    lib = ctypes.CDLL(gw.LIB_PATH)
    lib.gw_k_qknorm_rope_store.argtypes = [P, I, I, I, I, I, P, P, P, P, P, P, P, P]
    lib.gw_k_attn_decode.argtypes = [P, I, I, I, F, P, P, P, I, P, P, P, I, I, P]
    lib.gw_k_attn_part.argtypes = [P, I, P, I, I, I, I, F, P, P, P, P, I, I, I, P]
    bf, nh, nkv = kvt == "bf16", 8, 2
    nb, scale, rng = pos // 256 + 1, hd ** -0.5, np.random.default_rng(pos + bf)
    # q is about 4 in every dim (rows near 1, norm weights 4, no rotation), so K = c in every dim gives the score 4 c sqrt(hd):
    # position 7's is 82 .. 100 above the others', the row's own 68
    low = rng.uniform(-100, -82, (nb, 256, nkv, 1))
    low[:, 7] = 0
    k = (low / (4 * hd ** 0.5) + rng.uniform(-1, 1, (nb, 256, nkv, hd)) * 0.01).astype(np.float32)
    v = rng.choice([-1.0, 1.0], (nb, 256, nkv, hd)) * 2.0 ** -rng.uniform(0, 24, (nb, 256, nkv, hd)) * rng.integers(0, 2, (nb, 256, nkv, hd))
    if bf:  # (a sixteenth of it denormal by itself)
        v = np.where(rng.integers(0, 16, v.shape) == 0, v * 2.0 ** -126, v)
    v[:, 7] = 0
    v = v.astype(np.float32)

    def bits(x, isv):
        b = np.ascontiguousarray((x.view(np.uint32) >> 16).astype(np.uint16) if bf else x.astype(np.float16).view(np.uint16))
        b.reshape(-1, nkv, hd)[pos:] = 0x7fc0 if bf else 0x7e00
        return torch.from_numpy(_tiles(b, bf, isv).view(np.int16)).cuda()
    K, V = bits(k, False), bits(v, True)
    row = np.concatenate([1 + rng.uniform(-0.01, 0.01, nh * hd), -1 + rng.uniform(-0.01, 0.01, nkv * hd), rng.uniform(0, 2e-7, nkv * hd)])
    qn, kn, rope = np.full(hd, 4, np.float32), np.full(hd, 17 * hd ** -0.5, np.float32), np.zeros((pos + 1, hd), np.float32)
    rope[:, :hd // 2] = 1
    row, qn, kn, rope = (torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda() for a in (row, qn, kn, rope))
    stride, ld = nb * (hd + 2), row.numel()

    def part():
        return torch.full((nh, stride), 3.0, device="cuda")
    got = {}
    K1, V1, got["decode"] = K.clone(), V.clone(), part()
    assert lib.gw_k_attn_decode(row.data_ptr(), nh, nkv, hd, scale, qn.data_ptr(), kn.data_ptr(), rope.data_ptr(), pos, K1.data_ptr(),
                                V1.data_ptr(), got["decode"].data_ptr(), stride, int(bf), None) == 0
    at = torch.tensor([pos], dtype=torch.int32, device="cuda")
    kt = torch.tensor([gw.RQ_KV_BF16 if bf else gw.RQ_KV_F16], dtype=torch.int32, device="cuda")
    kp, vp = (torch.tensor([x.data_ptr()], dtype=torch.int64, device="cuda") for x in (K, V))
    assert lib.gw_k_qknorm_rope_store(row.data_ptr(), ld, 1, nh, nkv, hd, qn.data_ptr(), kn.data_ptr(), rope.data_ptr(), at.data_ptr(),
                                      kp.data_ptr(), vp.data_ptr(), kt.data_ptr(), None) == 0
    items = torch.tensor([[0, 1, g, b] for b in range(nb) for g in range(nkv)], dtype=torch.int32, device="cuda")
    for narrow in (0, 1):
        got["narrow" if narrow else "rows"] = part()
        assert lib.gw_k_attn_part(items.data_ptr(), len(items), row.data_ptr(), ld, nh, nkv, hd, scale, at.data_ptr(), kp.data_ptr(),
                                  vp.data_ptr(), got["narrow" if narrow else "rows"].data_ptr(), stride, int(bf), narrow, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(K, K1) and torch.equal(V, V1)
    kh, vh, q = K.cpu().numpy(), V.cpu().numpy(), row.cpu().numpy()
    f = orc.lib().or_attention_block_bf16 if bf else orc.lib().or_attention_block

    def oracle():
        o = np.zeros((nh, nb, hd + 2), np.float32)
        for h in range(nh):
            for b in range(nb):
                f(o[h, b].ctypes.data, o[h, b, hd:].ctypes.data, q[h * hd:].ctypes.data, kh.ctypes.data, vh.ctypes.data, pos + 1, b,
                  h // (nh // nkv), nkv, hd, scale)
        return o.reshape(nh, stride).view(np.uint32)
    kept = oracle()
    assert torch.set_flush_denormal(True)
    try:
        want = oracle()
    finally:
        torch.set_flush_denormal(False)
    assert (kept != want).mean() > 0.2  # (the modes decide these bits)
    # (+ 0: where a chain ends on -0, the zero products behind the row's positions make it +0 on the matrix cores. The combine's
    # sums start at +0 and the quantizer gives either zero the code 0, so no result of a pass has that sign)
    for name, x in got.items():
        assert _bits_equal(x.cpu().numpy() + np.float32(0), want.view(np.float32) + np.float32(0)), name
