"""GPU parity of the decode attention whose keys are split over workgroups
(long contexts) with the one-launch form and an fp64 restatement, and of a
DecodeGraph that crosses from one form to the other."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _split_always(monkeypatch):
    from parrot import hip_moe
    monkeypatch.setattr(hip_moe, "decode_splits", lambda context, batch, window=None:
                        context is not None)
    monkeypatch.setattr(hip_moe, "decode_split_line", lambda *shape: 0)
    return hip_moe


def _local_inputs(b, H, Hk, d, max_pos, seed):
    g = torch.Generator().manual_seed(seed)
    shapes = ((b, H, 1, d), (b, Hk, 1, d), (b, Hk, 1, d), (b, Hk, max_pos, d),
              (b, Hk, max_pos, d))
    return [torch.randn(s, generator=g).bfloat16().cuda() for s in shapes]


def _attend64(q, keys, values, scale):
    """q [b, H, d] over keys / values [b, Hk, L, d], fp64."""
    rep = q.shape[1] // keys.shape[1]
    k, v = (t.double().repeat_interleave(rep, 1) for t in (keys, values))
    s = torch.matmul(k, q.double().unsqueeze(-1)).squeeze(-1) * scale
    return torch.matmul(s.softmax(-1).unsqueeze(-2), v).squeeze(-2)


# chunk edges (64 keys), the window's edge, head groups of 1 to 16, every
# head width the split form takes, one -inf chunk
@pytest.mark.parametrize("b,H,Hk,d,max_pos,window,position,masked", [
    (1, 8, 2, 96, 256, 200, 0, None), (2, 8, 2, 96, 256, 200, 63, None),
    (1, 8, 2, 96, 256, 200, 64, None), (3, 8, 2, 96, 256, 200, 255, None),
    (2, 6, 6, 64, 300, 100, 130, None), (1, 16, 1, 128, 700, 700, 699, None),
    (2, 6, 2, 32, 513, 400, 512, None), (1, 4, 2, 192, 300, 300, 191, None),
    (1, 2, 1, 256, 300, 300, 299, None), (3, 12, 1, 96, 300, 300, 129, None),
    (1, 8, 2, 96, 4096, 4096, 4000, None), (1, 8, 2, 96, 300, 300, 250, (64, 128)),
    (1, 8, 2, 96, 300, 300, 250, (0, 190))])
def test_split_decode_attention(monkeypatch, b, H, Hk, d, max_pos, window, position, masked):
    hip_moe = _split_always(monkeypatch)
    print(f"split decode b={b} H={H}/{Hk} d={d} p={position} window={window}", flush=True)
    q, kn, vn, kc, vc = _local_inputs(b, H, Hk, d, max_pos, position + d)
    if masked is not None:  # positive queries against -inf keys: scores of -inf
        q = q.abs() + 0.125
        kc[:, :, masked[0]:masked[1]] = float("-inf")
    pos = torch.tensor([position], dtype=torch.int32, device="cuda")
    dim, scale = 512, d ** -0.5
    w = (torch.randn(dim, H * d, device="cuda") * (H * d) ** -0.5).bfloat16()
    caches = [(kc.clone(), vc.clone()) for _ in range(3)]
    with torch.no_grad():
        one = hip_moe.decode_attention(q, kn, vn, *caches[0], pos, window, scale)
        got = hip_moe.decode_attention(q, kn, vn, *caches[1], pos, window, scale,
                                       context=position + 1)
        heads = hip_moe.decode_attention_heads(q, kn, vn, *caches[2], pos, window, scale, w,
                                               context=position + 1)
    for k, v in caches:  # the new rows stored, every other row untouched
        kc[:, :, position], vc[:, :, position] = kn[:, :, 0], vn[:, :, 0]
        assert torch.equal(k, kc) and torch.equal(v, vc)
    lo = max(0, position - window + 1)
    ref = _attend64(q[:, :, 0], kc[:, :, lo:position + 1], vc[:, :, lo:position + 1], scale)
    got64 = got.double().view(b, H, d)
    # one bf16 rounding plus fp32 reassociation, as for the one-launch form
    assert ((got64 - ref).abs() <= 2 ** -8 * ref.abs().max() + 1e-5).all()
    assert ((one.double().view(b, H, d) - got64).abs() <= 2 ** -7 * ref.abs().max()).all()
    # each head's contribution: the bf16 output times its weight slice
    per_head = w.double().view(dim, H, d)
    want = torch.stack([got64[:, h] @ per_head[:, h].T for h in range(H)], 1)
    size = torch.stack([got64[:, h].abs() @ per_head[:, h].abs().T for h in range(H)], 1)
    assert ((heads.double() - want).abs() <= 1e-6 * size + 1e-7).all()


# the default layers on either side of their line, past the window, and a shape
# with a line of its own
@pytest.mark.parametrize("b,H,Hk,d,contexts", [
    (1, 8, 2, 96, (352, 353, 2500)), (8, 8, 2, 96, (576, 577, 3002)), (2, 8, 8, 96, (768, 769))])
def test_split_decode_attention_at_its_line(b, H, Hk, d, contexts):
    """With the rule as it is: the contexts past the line take a workspace, and
    all agree with the one-launch form as in the tests above."""
    from parrot import hip_moe
    max_pos, window, first = 4096, 2048, contexts[1]
    for context in contexts:
        print(f"split decode b={b} H={H}/{Hk} context {context}", flush=True)
        assert (hip_moe.decode_split_bytes(b, H, Hk, d, max_pos, window, context) > 0) == (context >= first)
        q, kn, vn, kc, vc = _local_inputs(b, H, Hk, d, max_pos, context)
        pos = torch.tensor([context - 1], dtype=torch.int32, device="cuda")
        caches = [(kc.clone(), vc.clone()) for _ in range(2)]
        with torch.no_grad():
            one, got = (hip_moe.decode_attention(q, kn, vn, *c, pos, window, d ** -0.5, context=known)
                        for c, known in zip(caches, (None, context)))
        assert all(torch.equal(x, y) for x, y in zip(*caches))
        if context < first:
            assert torch.equal(one, got)
        assert ((one.double() - got.double()).abs() <= 2 ** -7 * one.double().abs().max()).all()


# the NaN key alone in the last chunk, beside others, and in a full first chunk
@pytest.mark.parametrize("position,nan_key", [(64, 64), (70, 70), (130, 5), (255, 255)])
def test_split_decode_attention_nan_key(monkeypatch, position, nan_key):
    """A NaN in a key reaches the outputs of the heads that read it, wherever
    the key falls among the chunks, as in the one-launch form."""
    hip_moe = _split_always(monkeypatch)
    print(f"split decode NaN key {nan_key} p={position}", flush=True)
    q, kn, vn, kc, vc = _local_inputs(1, 8, 2, 96, 256, position)
    (kn[:, 0, 0] if nan_key == position else kc[:, 0, nan_key])[:, 3] = float("nan")
    pos = torch.tensor([position], dtype=torch.int32, device="cuda")
    with torch.no_grad():
        one, got = (hip_moe.decode_attention(q, kn, vn, kc.clone(), vc.clone(), pos, 256,
                                             96 ** -0.5, context=context)
                    for context in (None, position + 1))
    for out in (one, got):
        rows = out.view(8, 96)
        assert rows[:4].isnan().all() and not rows[4:].isnan().any()


@pytest.mark.parametrize("b,H,r,position", [(1, 8, 128, 0), (2, 8, 128, 64), (3, 6, 128, 700),
                                            (1, 16, 64, 129), (2, 3, 32, 383)])
def test_split_decode_attention_latent(monkeypatch, b, H, r, position):
    """fp32 queries (three bf16 parts in the score product) stay fp32 exact:
    no further from fp64 than the one-launch fp32 dot, within 1e-6."""
    hip_moe = _split_always(monkeypatch)
    print(f"split latent b={b} H={H} r={r} p={position}", flush=True)
    g = torch.Generator().manual_seed(position + r)
    max_pos = 800
    q = (torch.randn(b, 1, H * r, generator=g) * 3).cuda()
    new = torch.randn(b, 1, r, generator=g).bfloat16().cuda()
    cache = torch.randn(b, max_pos, r, generator=g).bfloat16().cuda()
    pos = torch.tensor([position], dtype=torch.int32, device="cuda")
    c1, c2 = cache.clone(), cache.clone()
    with torch.no_grad():
        one = hip_moe.decode_attention_latent(q, new, c1, pos, H, 96 ** -0.5)
        got = hip_moe.decode_attention_latent(q, new, c2, pos, H, 96 ** -0.5,
                                              context=position + 1)
    cache[:, position] = new[:, 0]
    assert torch.equal(c1, cache) and torch.equal(c2, cache)
    keys = cache[:, None, :position + 1]
    ref = _attend64(q.view(b, H, r), keys, keys, 96 ** -0.5).view(b, -1)
    err = [float((x.double() - ref).norm() / ref.norm()) for x in (one, got)]
    print("  relative error", err, flush=True)
    assert err[1] <= max(1e-6, 1.5 * err[0])


@pytest.mark.parametrize("b,r,position,size", [(1, 128, 352, 1), (4, 128, 500, 3), (2, 64, 1000, 1),
                                               (4, 128, 2000, 0.25), (1, 256, 600, 1)])
def test_split_decode_attention_latent_is_no_further_from_fp64(monkeypatch, b, r, position, size):
    """Pooled over 16 draws (the ratio of two such errors varies by about 5 %)
    the split form's error against fp64 is no larger than the one-launch
    form's."""
    hip_moe = _split_always(monkeypatch)
    print(f"split latent error b={b} r={r} p={position} size={size}", flush=True)
    H, square = 8, [0.0, 0.0]
    pos = torch.tensor([position], dtype=torch.int32, device="cuda")
    for seed in range(16):
        g = torch.Generator(device="cuda").manual_seed(seed)
        q = torch.randn(b, 1, H * r, generator=g, device="cuda") * size
        new = torch.randn(b, 1, r, generator=g, device="cuda").bfloat16()
        cache = torch.randn(b, position + 1, r, generator=g, device="cuda").bfloat16()
        with torch.no_grad():
            outs = [hip_moe.decode_attention_latent(q, new, cache, pos, H, 96 ** -0.5, context=context)
                    for context in (None, position + 1)]
        keys = cache[:, None]  # the new latent stored at its position
        ref = _attend64(q.view(b, H, r), keys, keys, 96 ** -0.5).view(b, -1)
        for i, out in enumerate(outs):
            square[i] += float(((out.double() - ref).norm() / ref.norm()) ** 2)
    print("  pooled relative errors", [(x / 16) ** 0.5 for x in square], flush=True)
    assert square[1] <= square[0]


# in the first chunk and beside the newest latent; queries that are bf16
# values (no later parts) and such that are not
@pytest.mark.parametrize("key", [5, 130])
@pytest.mark.parametrize("rounded", [True, False])
def test_split_decode_attention_latent_infinite(monkeypatch, key, rounded):
    """An infinite latent entry takes its key out of the softmax (score -inf)
    or makes the head NaN (score +inf), as in the one-launch form."""
    hip_moe = _split_always(monkeypatch)
    print(f"split latent infinite key {key} rounded={rounded}", flush=True)
    b, H, r, position, dim = 1, 8, 128, 130, 3
    g = torch.Generator().manual_seed(key)
    q = torch.randn(b, 1, H, r, generator=g)
    q[..., dim] = q[..., dim].abs() + 0.25
    q[:, :, H // 2:, dim] *= -1  # heads that see -inf, then heads that see +inf
    q = (q.bfloat16().float() if rounded else q).view(b, 1, H * r).cuda()
    new = torch.randn(b, 1, r, generator=g).bfloat16().cuda()
    cache = torch.randn(b, 200, r, generator=g).bfloat16().cuda()
    (new[:, 0] if key == position else cache[:, key])[:, dim] = float("-inf")
    pos = torch.tensor([position], dtype=torch.int32, device="cuda")
    with torch.no_grad():
        one, got = (hip_moe.decode_attention_latent(q, new, cache.clone(), pos, H, 96 ** -0.5,
                                                    context=context).view(H, r)
                    for context in (None, position + 1))
    for out in (one, got):  # weight 0 times an infinite value: that dimension alone
        finite = torch.isfinite(out)
        assert finite[:H // 2, :dim].all() and finite[:H // 2, dim + 1:].all()
        assert not finite[:, dim].any() and not finite[H // 2:].any()
    keep = torch.isfinite(one)
    assert ((one - got).abs()[keep] <= 1e-5).all()  # fp32 sums of ~130 terms of size 1


@pytest.mark.parametrize("logits", [False, True])
def test_decode_graph_crosses_into_the_split_form(logits):
    """Steps on either side of the position from which the keys are split
    equal eager steps, and the graph's output stays the same tensor."""
    from parrot import ModelConfig, Parrot, hip_moe
    from parrot.decode_graph import DecodeGraph
    # four heads per key row and rows of 96 and 128: shapes that split at the first
    # line (four heads of 64 on two would not below 2000 keys)
    cfg = ModelConfig(vocab_size=512, dim=256, n_layers=4, n_heads=8, n_kv_heads=2, head_dim=96,
                      kv_latent_dim=128, window_size=512, max_seq_len=512, n_experts=4,
                      expert_dim=64, shared_expert_dim=64, moe_backend="grouped_hip",
                      depth_backend="hip", collect_router_stats=False)
    torch.manual_seed(3)
    model = Parrot(cfg).to(device="cuda", dtype=torch.bfloat16).eval()
    first = next(p for p in range(1, 500) if hip_moe.decode_splits(p + 1, 2))
    prompt = torch.randint(0, 512, (2, first - 2), device="cuda")
    _, state = model.prefill(prompt)
    _, eager = model.prefill(prompt)
    graph = DecodeGraph(model, state, logits=logits)
    ids, out = prompt[:, -1:].clone(), graph.out
    for step in range(5):
        got = graph.step(ids)
        assert got.data_ptr() == out.data_ptr()
        want, _ = (model.decode_step if logits else model.decode_next)(ids, eager)
        assert torch.equal(got, want), f"step {step} at position {eager.position - 1}"
        ids = (got.argmax(-1) if logits else got).clone()
    assert set(graph.graphs) == {False, True}
    with torch.inference_mode():
        graph._rewind(first - 1)  # back to the one-launch form: no new capture
    graph.step(ids)
    assert len(graph.graphs) == 2 and state.position == first


def _long_model(**fields):
    from parrot import ModelConfig, Parrot
    cfg = ModelConfig(**{**dict(vocab_size=512, dim=256, n_layers=4, n_heads=8, n_kv_heads=2,
                                head_dim=96, kv_latent_dim=128, window_size=512, max_seq_len=512,
                                n_experts=4, expert_dim=64, shared_expert_dim=64,
                                moe_backend="grouped_hip", depth_backend="hip",
                                collect_router_stats=False), **fields})
    torch.manual_seed(3)
    return Parrot(cfg).to(device="cuda", dtype=torch.bfloat16).eval()


# (max_seq_len, prompt): ends below the line, crosses it, starts past it
@pytest.mark.parametrize("limit,start,forms", [(300, 40, {False}), (512, 40, {False, True}),
                                               (512, 400, {True})])
def test_decode_graph_captures_up_front(monkeypatch, limit, start, forms):
    """Every form that the generation comes to is captured when the graph is
    made, in one pool; no step captures, and a state set back below the line
    goes on with what there is."""
    from parrot.decode_graph import DecodeGraph
    print(f"decode graph forms, {start} to {limit}", flush=True)
    model = _long_model(max_seq_len=limit)
    prompt = torch.randint(0, 512, (2, start), device="cuda")
    _, state = model.prefill(prompt)
    graph = DecodeGraph(model, state)
    assert set(graph.graphs) == forms and state.position == start
    assert int(state.position_device) == start
    assert len({g.pool() for g in graph.graphs.values()}) == 1
    assert graph.graph is graph.graphs[start == 400]  # the next step's
    monkeypatch.setattr(torch.cuda, "graph", None)
    for position in (limit - 1, start):
        with torch.inference_mode():
            graph._rewind(position)
        graph.step(prompt[:, -1:].clone())
    assert state.position == start + 1


# widths without a split kernel, and a line past the longest context
@pytest.mark.parametrize("fields", [dict(head_dim=16, kv_latent_dim=16),
                                    dict(head_dim=64, kv_latent_dim=64)])
def test_decode_graph_of_a_shape_that_never_splits(fields):
    from parrot.decode_graph import DecodeGraph
    print(f"decode graph {fields}", flush=True)
    model = _long_model(**fields)
    _, state = model.prefill(torch.randint(0, 512, (1, 400), device="cuda"))
    assert set(DecodeGraph(model, state).graphs) == {False}


def test_decode_graph_between_two_lines():
    """Layers that split from different positions: the second form begins
    where the last of them does, and steps equal eager ones on both sides."""
    import copy
    from parrot.decode_graph import DecodeGraph
    print("decode graph, local line 545, latent line 353", flush=True)
    model = _long_model(n_kv_heads=8, window_size=1024, max_seq_len=1024)
    prompt = torch.randint(0, 512, (1, 541), device="cuda")
    with torch.inference_mode():
        _, state = model.prefill(prompt)
        other = copy.deepcopy(state)
        graph = DecodeGraph(model, state)
        assert set(graph.graphs) == {False, True} and graph._line == 544
        mine = theirs = prompt[:, -1:].clone()
        for _ in range(6):
            mine = graph.step(mine)
            theirs, other = model.decode_next(theirs, other)
            assert torch.equal(mine, theirs)


# the eager step, the first capture and the second one
@pytest.mark.parametrize("fails_at", [1, 2, 3])
def test_decode_graph_that_fails_leaves_the_state(monkeypatch, fails_at):
    """A constructor that raises has taken no step: eager decoding goes on
    from the same position with the same tokens."""
    import copy
    from parrot.decode_graph import DecodeGraph
    print(f"decode graph failing at run {fails_at}", flush=True)
    model = _long_model()
    prompt = torch.randint(0, 512, (2, 40), device="cuda")
    with torch.inference_mode():
        _, state = model.prefill(prompt)
        other = copy.deepcopy(state)
        runs, run = [], DecodeGraph._run

        def failing(self):
            runs.append(run(self))
            if len(runs) == fails_at:
                raise RuntimeError("planted on the host")
            return runs[-1]
        monkeypatch.setattr(DecodeGraph, "_run", failing)
        with pytest.raises(RuntimeError, match="planted"):
            DecodeGraph(model, state)
        assert len(runs) == fails_at and state.position == 40 and int(state.position_device) == 40
        mine = theirs = prompt[:, -1:]
        for _ in range(3):
            mine, theirs = model.decode_next(mine, state)[0], model.decode_next(theirs, other)[0]
            assert torch.equal(mine, theirs)


def test_decode_graph_logits_are_written_in_place(monkeypatch):
    """Both forms' captured steps end in the same output tensor, with no copy
    behind the vocabulary product."""
    from parrot import hip_moe
    from parrot.decode_graph import DecodeGraph
    print("decode graph logits in place", flush=True)
    outs, logits = [], hip_moe.vocab_logits

    def recorded(h, weight, out=None):
        outs.append(logits(h, weight, out))
        return outs[-1]
    monkeypatch.setattr(hip_moe, "vocab_logits", recorded)
    model = _long_model()
    _, state = model.prefill(torch.randint(0, 512, (2, 40), device="cuda"))
    del outs[:]
    graph = DecodeGraph(model, state, logits=True)
    assert len(outs) == 3 and len(graph.graphs) == 2  # the eager step, then the captured ones
    assert all(o.data_ptr() == graph.out.data_ptr() and o.shape == (2, 1, 512) for o in outs[1:])
    h = torch.randn(2, 1, 256, device="cuda").bfloat16()
    with torch.no_grad():
        want = logits(h, model.embedding.weight)
        out = torch.empty_like(want)
        assert logits(h, model.embedding.weight, out) is out and torch.equal(out, want)
        for bad in (out[:1], out.double(), out.cpu(), out.transpose(0, 1)):
            with pytest.raises(RuntimeError, match="contiguous fp32"):
                logits(h, model.embedding.weight, bad)
