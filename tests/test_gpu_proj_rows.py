"""GPU parity of the projections over many rows (32- and 64-row tiles, all
columns streamed) with the 16-row kernel, which the same rows take in chunks:
a row's outputs do not depend on how many rows a call has, so they must agree
bit for bit, and with fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CHUNK = 480  # rows that take the 16-row kernel; whole 32-key blocks


def _operands(rows, k, n, seed, pad=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(rows, k + pad, generator=g, device="cuda").bfloat16()[:, :k]
    w = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).bfloat16()
    from parrot import hip_moe
    return x, w, hip_moe._fragment_order(w)


@pytest.mark.parametrize("rows,k,n,with_addend,pad", [
    (1100, 768, 768, True, 0), (2047, 768, 896, False, 0), (4096, 512, 64, True, 0),
    (4097, 768, 768, True, 0), (4200, 128, 1536, False, 768), (5001, 256, 16, True, 8),
    (1729, 768, 80, True, 0), (9000, 768, 1152, False, 0),
    # few columns and short k loops change over later: a partial last block of
    # 16 columns, one block and a part, two, and ten with an addend
    (1500, 768, 784, True, 0), (24001, 768, 80, True, 8), (37000, 512, 64, False, 0),
    (9001, 256, 512, True, 0)])
def test_proj_rows(rows, k, n, with_addend, pad):
    from parrot import hip_moe
    print(f"proj rows={rows} k={k} n={n} addend={with_addend} pad={pad}", flush=True)
    x, w, packed = _operands(rows, k, n, rows + n, pad)
    add = torch.randn(rows, n, device="cuda").bfloat16() if with_addend else None
    with torch.no_grad():
        got = hip_moe.proj(x, packed, n, addend=add)
        parts = [hip_moe.proj(x[i:i + CHUNK], packed, n,
                              addend=None if add is None else add[i:i + CHUNK])
                 for i in range(0, rows, CHUNK)]
    assert torch.equal(got, torch.cat(parts))
    ref = x.float() @ w.float().T
    bound = 1e-6 * k * (x.float().abs() @ w.float().abs().T) + 2 ** -8 * ref.abs()
    if add is not None:  # the sum is rounded once more
        ref = ref + add.float()
        bound = bound + 2 ** -8 * ref.abs()
    assert ((got.float() - ref).abs() <= bound).all()


def _tables(positions, d):
    i = torch.arange(0, d, 2, device="cuda").float()
    angle = torch.arange(positions, device="cuda").float()[:, None] * 10000.0 ** (-i / d)
    return angle.cos().contiguous(), angle.sin().contiguous()


def _valid(frag, t, d):
    """The 32-key blocks of fragment-order K or V that hold no padding key."""
    return frag.view(frag.shape[0], frag.shape[1], -1, 32 * d)[:, :, :t // 32]


# ragged ends, head widths that straddle the 48-column blocks, one and several
# sequences, both tile heights, with and without row-major copies
@pytest.mark.parametrize("b,t,heads,kv,d,dim,cache", [
    (3, 333, 8, 2, 96, 768, True), (1, 1025, 8, 2, 96, 768, False), (2, 2047, 8, 2, 96, 768, True),
    (5, 258, 4, 4, 64, 512, True), (9, 513, 6, 3, 128, 256, True), (1, 4500, 4, 1, 64, 768, True)])
def test_proj_rope_qkv_rows(b, t, heads, kv, d, dim, cache):
    from parrot import hip_moe
    print(f"proj rope rows b={b} t={t} heads={heads}/{kv} d={d} dim={dim}", flush=True)
    n = (heads + 2 * kv) * d
    x, _, packed = _operands(b * t, dim, n, t + n)
    x = x.view(b, t, dim)
    cos, sin = _tables(t + 8, d)
    with torch.no_grad():
        q, kf, vf, k, v = hip_moe.proj_rope_qkv_frag(x, packed, cos, sin, heads, kv, d,
                                                     cache_kv=cache)
        # row-major and transposed values through the other entry, from position 5
        q5, k5, v5 = hip_moe.proj_rope_qkv(x, packed, cos, sin, heads, kv, d, start=5)
        vt = hip_moe.proj_rope_qkv(x, packed, cos, sin, heads, kv, d, vt_keys=(t + 35) // 4 * 4)[2]
        for n_b in range(b):
            for at in range(0, t, CHUNK):
                end = min(t, at + CHUNK)
                piece = x[n_b:n_b + 1, at:end]
                rq, rk, rv = hip_moe.proj_rope_qkv(piece, packed, cos, sin, heads, kv, d, start=at)
                assert torch.equal(q[n_b, :, at:end], rq[0])
                if cache:
                    assert torch.equal(k[n_b, :, at:end], rk[0])
                    assert torch.equal(v[n_b, :, at:end], rv[0])
                assert torch.equal(vt[n_b, :, :, at:end], rv[0].transpose(-1, -2))
                pk, pv = hip_moe.pack_kv_fragments(rk, rv)
                lo, cnt = at // 32, (end - at) // 32
                assert torch.equal(_valid(kf, t, d)[n_b, :, lo:lo + cnt], _valid(pk, end - at, d)[0])
                assert torch.equal(_valid(vf, t, d)[n_b, :, lo:lo + cnt], _valid(pv, end - at, d)[0])
                if end == t and t % 32:  # the last block's valid keys, through the attention's order
                    tail_k, tail_v = (z.view(*z.shape[:2], -1, 32 * d)[n_b, :, -1] for z in (kf, vf))
                    want_k, want_v = (z.view(1, kv, -1, 32 * d)[0, :, -1] for z in (pk, pv))
                    keep_k, keep_v = hip_moe.pack_kv_fragments(
                        *(torch.ones(1, kv, t % 32, d, device="cuda", dtype=torch.bfloat16)
                          for _ in range(2)))
                    for got, want, keep in ((tail_k, want_k, keep_k), (tail_v, want_v, keep_v)):
                        keep = keep.view(kv, 32 * d) == 1
                        assert torch.equal(got[keep], want[keep])
                r5 = hip_moe.proj_rope_qkv(piece, packed, cos, sin, heads, kv, d, start=at + 5)
                assert all(torch.equal(z[n_b, :, at:end], w[0]) for z, w in zip((q5, k5, v5), r5))


@pytest.mark.parametrize("b,t,heads,d,r", [(1, 1024, 8, 96, 128), (3, 333, 8, 96, 128),
                                           (2, 2049, 4, 64, 256), (9, 500, 2, 128, 128)])
def test_proj_kv_fragments_rows(b, t, heads, d, r):
    """[Wk; Wv] from a row-strided latent, and each map alone."""
    from parrot import hip_moe
    print(f"proj kv rows b={b} t={t} heads={heads} d={d} r={r}", flush=True)
    n = heads * d
    x, w, packed = _operands(b * t, r, 2 * n, t + r, pad=64)
    x = x.view(b, t, r)
    with torch.no_grad():
        kf, vf = hip_moe.proj_kv_frag(x, packed, n, d)
        alone = [hip_moe.proj_frag(x, hip_moe._fragment_order(m.contiguous()), n, d, values)
                 for m, values in ((w[:n], False), (w[n:], True))]
        for got, one in zip((kf, vf), alone):
            assert torch.equal(_valid(got, t, d), _valid(one, t, d))
        for n_b in range(b):
            for at in range(0, t, CHUNK):
                end = min(t, at + CHUNK)
                rk, rv = hip_moe.proj_kv_frag(x[n_b:n_b + 1, at:end], packed, n, d)
                lo, cnt = at // 32, (end - at) // 32
                assert torch.equal(_valid(kf, t, d)[n_b, :, lo:lo + cnt], _valid(rk, end - at, d)[0])
                assert torch.equal(_valid(vf, t, d)[n_b, :, lo:lo + cnt], _valid(rv, end - at, d)[0])
