"""Host-side rules that pick a kernel, and the argument checks of their C
entry points (no GPU)."""
import ctypes


def test_decode_split_rule():
    from parrot import hip_moe
    assert not hip_moe.decode_splits(None, 1)
    assert not hip_moe.decode_splits(352, 1) and hip_moe.decode_splits(353, 1)
    assert not hip_moe.decode_splits(4096, 1, window=352)  # the window bounds the keys
    assert not hip_moe.decode_splits(1024, 64) and hip_moe.decode_splits(1025, 64)


def test_decode_split_arguments():
    from parrot import _abi
    lib, fake, null = _abi.load(), ctypes.c_void_p(4096), None
    size = lib.parrot_decode_attention_split_workspace_bytes
    # (max, sum) pairs and partial rows of 32 chunks of 64 keys
    assert size(1, 8, 2, 96, 4096, 2048) == 8 * 32 * 8 + 8 * 32 * 96 * 4
    assert size(1, 8, 2, 16, 4096, 2048) == 0 and size(1, 34, 2, 96, 4096, 2048) == 0
    assert size(1, 8, 3, 96, 4096, 2048) == 0

    def local(q=4096, heads=8, d=96, ws=4096, wsb=1 << 20, out=fake):
        return lib.parrot_decode_attention_split_bf16(
            q, fake, fake, fake, fake, fake, 1, heads, 2, d, 4096, 2048, 0.1, out, ws, wsb, null)
    assert local(q=null) == -1 and local(out=null) == -1
    assert local(heads=7) == -3 and local(d=16) == -3 and local(heads=34) == -3
    assert local(ws=null) == -4 and local(wsb=64) == -4
    assert local(q=4096 + 8) == -5 and local(ws=4096 + 8) == -5

    def heads(dim=768, w=fake, wsb=1 << 20):
        return lib.parrot_decode_attention_heads_split_bf16(
            fake, fake, fake, fake, fake, fake, 1, 8, 2, 96, 4096, 2048, 0.1, w, dim, fake, fake,
            wsb, null)
    assert heads(w=null) == -1 and heads(dim=0) == -2 and heads(dim=776) == -3
    assert heads(wsb=64) == -4

    def latent(q=fake, r=128, wsb=1 << 22):
        return lib.parrot_decode_attention_latent_split_f32(
            q, fake, fake, fake, 1, 8, r, 4096, 0.1, fake, fake, wsb, null)
    assert latent(q=null) == -1 and latent(r=100) == -3 and latent(wsb=64) == -4


def test_decode_graph_forms():
    """The forms a generation comes to, known when its graph is made: none is
    left to a step, and none is captured that no layer takes."""
    from parrot.decode_graph import split_forms
    assert split_forms(128, 4096, 352) == [(False, 128), (True, 4095)]
    assert split_forms(351, 4096, 352) == [(False, 351), (True, 4095)]
    assert split_forms(352, 4096, 352) == [(True, 352)]
    assert split_forms(128, 352, 352) == [(False, 128)]
    assert split_forms(128, 353, 352) == [(False, 128), (True, 352)]
    assert split_forms(2000, 4096, None) == [(False, 2000)]


def test_decode_split_bytes_by_shape():
    from parrot import hip_moe
    size = hip_moe.decode_split_bytes
    assert size(1, 8, 2, 96, 4096, 2048, 353) > 0 and size(1, 8, 2, 96, 4096, 2048, 352) == 0
    assert size(1, 8, 2, 96, 4096, 256, 4096) == 0  # the window stays below the line
    assert size(1, 8, 2, 16, 4096, 2048, 4096) == 0 and size(1, 34, 2, 96, 4096, 2048, 4096) == 0
    assert size(1, 8, 2, 96, 4096, 2048, None) == 0


def test_decode_split_line_by_shape():
    """The default layers' line, whatever the batch, and later ones where fewer
    heads share a key row, rows are short, or the pairs are many."""
    from parrot import hip_moe
    size, line = hip_moe.decode_split_bytes, hip_moe.decode_split_line
    for b in (1, 2, 8, 22, 23, 64):
        first = next(c for c in range(1, 2049) if hip_moe.decode_splits(c, b))
        for shape in ((8, 2, 96, 4096, 2048), (8, 1, 128, 4096, 4096)):
            assert size(b, *shape, first) > 0 and size(b, *shape, first - 1) == 0
    assert size(1, 8, 8, 96, 4096, 4096, 544) == 0 and size(1, 8, 8, 96, 4096, 4096, 545) > 0
    assert size(8, 32, 32, 128, 4096, 4096, 4096) == 0  # 256 pairs fill the chip
    assert size(2, 4, 2, 64, 4096, 4096, 1984) == 0 and size(2, 4, 2, 64, 4096, 4096, 1985) > 0
    assert line(1, 16, 1, 128) == 384 and line(4, 32, 8, 128) == 832
