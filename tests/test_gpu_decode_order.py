"""Decode attention in an order of its own (ops.decode_seq_order): a permutation, longest first, and the bits of the launch without it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(s, nq, nkv, hd, bound, dev, seed=0):
    g = torch.Generator().manual_seed(seed)
    lens = torch.randint(0, bound + 1, (s,), generator=g, dtype=torch.int32)
    lens[0], lens[s // 2] = bound, 0
    cols = (bound + 15) // 16
    nb = 64 + cols
    bt = torch.randint(0, nb, (s, cols), generator=g, dtype=torch.int32).to(dev)
    kv = torch.randn(2, nb, 16, nkv, hd, generator=g).to(torch.bfloat16).to(dev)
    q = torch.randn(s, nq * hd, generator=g).to(torch.bfloat16).to(dev)
    return q, kv[0], kv[1], bt, lens.to(dev)


# launches of more than 256 workgroups: lone waves, two partitions, partitions that merge in their workgroup, a last round that is not full,
# more rounds than are resident, up to 1024 sequences
@pytest.mark.parametrize("s,nq,nkv,hd,bound", [(65, 28, 4, 128, 700), (120, 28, 4, 128, 700), (70, 28, 4, 128, 1000), (161, 32, 8, 128, 300), (257, 14, 2, 128, 320),
                                               (200, 32, 8, 128, 512), (300, 14, 2, 128, 600), (1024, 8, 1, 128, 520), (33, 40, 10, 128, 400)])
def test_order(s, nq, nkv, hd, bound):
    from vllm_omni_amd import ops

    dev = torch.device("cuda", 0)
    q, kc, vc, bt, lens = _case(s, nq, nkv, hd, bound, dev)
    order = ops.decode_seq_order(lens, nq, nkv, hd, 16, bound)
    if order is None:      # three partitions or more
        assert -(-bound // ops.decode_auto_partition(s, nkv, bound, 16, head_dim=hd)) > 2
        pytest.skip("not ordered at these sizes")
    assert torch.equal(order[0], lens)
    assert torch.equal(order[1].sort().values, torch.arange(s, dtype=torch.int32, device=dev))
    ps = ops.decode_auto_partition(s, nkv, bound, 16, head_dim=hd)
    ws = ops.new_decode_workspace(max(ops.decode_workspace_bytes(s, nq, hd, bound, ps), 16), dev)
    for kw in ({}, {"slopes": torch.rand(nq, device=dev), "sinks": torch.randn(nq, device=dev), "out_scale": 0.8}):
        want = ops.paged_attn_decode(torch.full_like(q, 7.0), q, kc, vc, bt, lens, bound, hd ** -0.5, workspace=ws, **kw)
        got = ops.paged_attn_decode(torch.full_like(q, 9.0), q, kc, vc, bt, lens, bound, hd ** -0.5, workspace=ws, order=order, **kw)
        assert torch.equal(want.view(torch.int16), got.view(torch.int16))


def test_longest_first():
    from vllm_omni_amd import ops

    dev = torch.device("cuda", 0)
    lens = torch.randint(1, 3000, (600,), dtype=torch.int32, device=dev)
    order = ops.decode_seq_order(lens, 32, 8, 128, 16, 3008)      # rounds of 32 sequences, five resident
    sorted_lens = lens.sort(descending=True).values
    for r in range(0, 600, 32):
        part = sorted_lens[r:r + 32]
        assert torch.equal(lens[order[1, r:r + 32].long()], part.flip(0) if r // 32 in (1, 3) else part)


def test_sizes_that_are_not_ordered():
    from vllm_omni_amd import ops

    dev = torch.device("cuda", 0)
    lens = lambda n: torch.full((n,), 100, dtype=torch.int32, device=dev)  # noqa: E731
    assert ops.decode_seq_order(lens(64), 28, 4, 128, 16, 2048) is None       # a workgroup a CU
    assert ops.decode_seq_order(lens(256), 28, 4, 128, 16, 256) is None       # short bounds
    assert ops.decode_seq_order(lens(512), 16, 2, 64, 16, 4096) is None
    assert ops.decode_seq_order(lens(1025), 8, 1, 128, 16, 2048) is None
    assert ops.decode_seq_order(lens(1), 28, 4, 128, 16, 2048) is None
    with pytest.raises(ValueError):
        q, kc, vc, bt, sl = _case(65, 28, 4, 128, 700, dev)
        ops.paged_attn_decode(torch.empty_like(q), q, kc, vc, bt, sl, 700, 0.1, order=torch.zeros(2, 64, dtype=torch.int32, device=dev))


def test_replays_follow_the_lengths():
    from vllm_omni_amd import ops

    dev = torch.device("cuda", 0)
    s, nq, nkv, hd, bound = 120, 28, 4, 128, 700
    q, kc, vc, bt, lens = _case(s, nq, nkv, hd, bound, dev)
    out = torch.empty_like(q)

    def step():
        order = ops.decode_seq_order(lens, nq, nkv, hd, 16, bound)
        return ops.paged_attn_decode(out, q, kc, vc, bt, lens, bound, hd ** -0.5, order=order)

    step()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step()
    for i in range(3):
        lens.copy_(torch.randint(0, bound + 1, (s,), dtype=torch.int32, generator=torch.Generator().manual_seed(i)))
        want = ops.paged_attn_decode(torch.empty_like(q), q, kc, vc, bt, lens, bound, hd ** -0.5)
        g.replay()
        assert torch.equal(want.view(torch.int16), out.view(torch.int16))


@pytest.mark.parametrize("lens,kept", [([700] * 120, True), ([660] * 60 + [700] * 60, True), ([600] * 60 + [700] * 60, False)])
def test_lengths_close_to_each_other_stay(lens, kept):
    from vllm_omni_amd import ops

    order = ops.decode_seq_order(torch.tensor(lens, dtype=torch.int32, device="cuda"), 28, 4, 128, 16, 700)
    assert torch.equal(order[1].cpu(), torch.arange(120, dtype=torch.int32)) == kept


# an order is a matter of speed: one made of other lengths gives the bits of the call's own
@pytest.mark.parametrize("biased", [False, True])
def test_an_order_of_other_lengths(biased):
    from vllm_omni_amd import ops

    dev = torch.device("cuda", 0)
    s, nq, nkv, hd, bound = 120, 28, 4, 128, 700
    q, kc, vc, bt, lens = _case(s, nq, nkv, hd, bound, dev)
    kw = {"slopes": torch.rand(nq, device=dev), "sinks": torch.randn(nq, device=dev)} if biased else {}
    order = ops.decode_seq_order(lens, nq, nkv, hd, 16, bound)
    lens = torch.randint(0, bound + 1, (s,), dtype=torch.int32, generator=torch.Generator().manual_seed(9)).to(dev)
    want = ops.paged_attn_decode(torch.empty_like(q), q, kc, vc, bt, lens, bound, hd ** -0.5, **kw)
    got = ops.paged_attn_decode(torch.empty_like(q), q, kc, vc, bt, lens, bound, hd ** -0.5, order=order, **kw)
    assert torch.equal(want.view(torch.int16), got.view(torch.int16))


# lengths below zero are empty sequences: the order is a permutation all the same, and nothing is written behind it
@pytest.mark.parametrize("s", [65, 67, 120, 129, 1023])
def test_lengths_below_zero(s):
    from vllm_omni_amd import _C, ops

    dev = torch.device("cuda", 0)
    lens = torch.randint(-3, 700, (s,), dtype=torch.int32, generator=torch.Generator().manual_seed(s))
    lens[:8] = torch.tensor([-2, -1, 0, -7, -(2 ** 31), 700, -2, -3])
    lens = lens.to(dev)
    room = torch.full((2 * s + 64,), 12345, dtype=torch.int32, device=dev)
    code = _C.lib.mi_decode_seq_order(room.data_ptr(), lens.data_ptr(), s, 28, 4, 128, 16, 700, 0, _C.MI_DECODE_PACKED_PV,
                                      torch.cuda.current_stream().cuda_stream)
    assert code == _C.MI_OK
    assert torch.equal(room[:s], lens)
    assert torch.equal(room[s:2 * s].sort().values, torch.arange(s, dtype=torch.int32, device=dev))
    assert (room[2 * s:] == 12345).all()
    order = ops.decode_seq_order(lens, 28, 4, 128, 16, 700)
    assert torch.equal(order.view(-1), room[:2 * s])


# the empty rows that fill a captured step up do not count as short contexts
@pytest.mark.parametrize("lens,kept", [([700] * 117 + [0] * 3, True), ([0] * 5 + [660] * 60 + [700] * 50 + [0] * 5, True), ([0] * 120, True),
                                       ([600] * 60 + [700] * 57 + [0] * 3, False), ([0] * 7 + [1] + [700] * 112, False)])
def test_empty_rows_do_not_count(lens, kept):
    from vllm_omni_amd import ops

    order = ops.decode_seq_order(torch.tensor(lens, dtype=torch.int32, device="cuda"), 28, 4, 128, 16, 700)
    assert torch.equal(order[1].cpu(), torch.arange(120, dtype=torch.int32)) == kept
    assert torch.equal(order[1].cpu().sort().values, torch.arange(120, dtype=torch.int32))


def _step(s, nq, nkv, bound, dtype, dev):
    """a decode step's rows: uneven contexts with this step's token in them, empty rows with slot -1, blocks of their own"""
    g = torch.Generator().manual_seed(s + bound)
    lens = torch.randint(0, bound + 1, (s,), generator=g, dtype=torch.int32)
    lens[0], lens[1], lens[s // 2], lens[s - 1] = bound, 1, 0, 0
    cols = (bound + 15) // 16
    table = (torch.randperm(s * cols, generator=g) + 1).view(s, cols).to(torch.int32)
    at = (lens.long() - 1).clamp(min=0)
    slots = torch.where(lens > 0, table[torch.arange(s), at // 16].long() * 16 + at % 16, -1)
    gd = torch.Generator(device=dev).manual_seed(s)
    kv = torch.randn(2, s * cols + 1, 16, nkv, 128, generator=gd, device=dev).to(dtype)
    rows = (nq + 2 * nkv) * 128
    norms = [(1 + 0.1 * torch.randn(128, generator=gd, device=dev)).to(dtype) for _ in range(2)]
    slabs = torch.randn(3, s, rows, generator=gd, device=dev)
    return lens.to(dev), table.to(dev), at.to(dev), slots.to(dev), kv, norms, slabs, torch.randn(rows, generator=gd, device=dev).to(dtype)


# the launches of a pure-decode step, which rotate, norm and write the token's cache row as well: outputs and caches
@pytest.mark.parametrize("slabs", [False, True], ids=["rows", "slabs"])
@pytest.mark.parametrize("norm", [False, True], ids=["plain", "qk-norm"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("s,nq,nkv,bound", [(120, 28, 4, 700), (70, 28, 4, 1000), (161, 32, 8, 300), (257, 14, 2, 320)])
def test_steps_that_write_the_cache(s, nq, nkv, bound, dtype, norm, slabs):
    from vllm_omni_amd import ops
    from vllm_omni_amd.layers import build_cos_sin_cache

    dev = torch.device("cuda", 0)
    lens, table, pos, slots, kv, norms, part, bias = _step(s, nq, nkv, bound, dtype, dev)
    order = ops.decode_seq_order(lens, nq, nkv, 128, 16, bound)
    assert order is not None and not torch.equal(order[1], torch.arange(s, dtype=torch.int32, device=dev))
    csc = build_cos_sin_cache(128, 2048, 1e6, device=dev)
    kw = dict(zip(("q_norm_weight", "k_norm_weight"), norms)) if norm else {}
    qkv = part[0].to(dtype)
    got = []
    for o in (None, order):
        cache = kv.clone()
        if slabs:
            p = ops.SplitKPartials(part, 3, s, qkv.shape[1], bias, dtype, (s,), dev, None)
            out = ops.rope_cache_paged_attn_decode_splitk(p, nq, nkv, 128, pos, csc, cache[0], cache[1], slots, table, lens, bound, 128 ** -0.5,
                                                          order=o, **kw)
        else:
            q, k, v = qkv.split([nq * 128, nkv * 128, nkv * 128], -1)
            out = torch.full((s, nq * 128), 7.0 if o is None else 9.0, dtype=dtype, device=dev)
            ops.rope_cache_paged_attn_decode(out, q, k, v, pos, csc, cache[0], cache[1], slots, table, lens, bound, 128 ** -0.5, order=o, **kw)
        got.append((out.view(torch.int16), cache.view(torch.int16)))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert not torch.equal(got[1][1], kv.view(torch.int16))


# partitions that merge behind their last arrival, by counters of (sequence, head group)
def test_fused_merge():
    from vllm_omni_amd import ops

    dev = torch.device("cuda", 0)
    s, nq, nkv, hd, bound = 70, 28, 4, 128, 1000
    q, kc, vc, bt, lens = _case(s, nq, nkv, hd, bound, dev)
    order = ops.decode_seq_order(lens, nq, nkv, hd, 16, bound)
    assert order is not None and -(-bound // ops.decode_auto_partition(s, nkv, bound, 16, head_dim=hd)) == 2
    want = ops.paged_attn_decode(torch.empty_like(q), q, kc, vc, bt, lens, bound, hd ** -0.5, fused_merge=False)
    ws = ops.new_decode_workspace(ops.decode_workspace_bytes(s, nq, hd, bound, ops.decode_auto_partition(s, nkv, bound, 16, head_dim=hd)), dev)
    for _ in range(2):      # the counters are back at zero
        got = ops.paged_attn_decode(torch.empty_like(q), q, kc, vc, bt, lens, bound, hd ** -0.5, workspace=ws, fused_merge=True, order=order)
        assert torch.equal(want.view(torch.int16), got.view(torch.int16))


# whole steps through the runner: 67 requests of uneven length, captured (filled up to 72 rows) and eager, with and without an order
@pytest.mark.parametrize("eager", [False, True], ids=["captured", "eager"])
@pytest.mark.parametrize("qk_norm", [False, True], ids=["plain", "qk-norm"])
def test_runner_steps(eager, qk_norm, monkeypatch):
    from vllm_omni_amd import ops
    from vllm_omni_amd.model_runner import GPUARModelRunner
    from vllm_omni_amd.sched_output import CachedRequestData, NewRequestData, SamplingParams, SchedulerOutput
    from vllm_omni_amd.talker import TalkerConfig

    dev = torch.device("cuda", 0)
    n, longest, steps = 67, 330, 4
    ctx = torch.randint(1, longest - steps, (n,), generator=torch.Generator().manual_seed(2)).tolist()
    per = (longest + 15) // 16
    made, real = [], ops.decode_seq_order

    def passes(ordered):
        def spy(*a, **k):
            o = real(*a, **k) if ordered else None
            made.append(o)
            return o

        monkeypatch.setattr(ops, "decode_seq_order", spy)
        c = TalkerConfig.from_json("mini_talker")
        c.mrope_section, c.head_dim, c.num_attention_heads, c.num_key_value_heads, c.qk_norm = None, 128, 8, 4, qk_norm
        r = GPUARModelRunner(c, dev, torch.bfloat16, max_num_reqs=128, max_model_len=longest, max_num_batched_tokens=128, block_size=16,
                             enforce_eager=eager, seed=0)
        r.load_model()
        r.initialize_kv_cache(n * per + 1)
        g = torch.Generator(device=dev).manual_seed(7)
        for kv in r.kv_caches:
            for x in kv:
                x.copy_(torch.randn(x.shape, generator=g, device=dev))
        ids, out = [f"r{i}" for i in range(n)], []
        for step in range(steps):
            sched = {i: 1 for i in ids}
            if step == 0:
                so = SchedulerOutput(scheduled_new_reqs=[NewRequestData(i, list(range(k + 1)), SamplingParams(temperature=0.0),
                                                                        (list(range(1 + j * per, 1 + (j + 1) * per)),), k)
                                                         for j, (i, k) in enumerate(zip(ids, ctx))],
                                     num_scheduled_tokens=sched, total_num_scheduled_tokens=n)
            else:
                so = SchedulerOutput(scheduled_cached_reqs=CachedRequestData(req_ids=ids, new_token_ids=[], new_block_ids=[None] * n,
                                                                             num_computed_tokens=[k + step for k in ctx], num_output_tokens=[step] * n),
                                     num_scheduled_tokens=sched, total_num_scheduled_tokens=n)
            r.execute_model(so)
            st = r.execute_model_state
            out += [st.logits[:n].clone(), st.hidden_states[:n].clone()]
            out.append(torch.tensor(r.sample_tokens().sampled_token_ids))
        return out + [x[1:].clone() for kv in r.kv_caches for x in kv]

    want = passes(False)
    made.clear()
    got = passes(True)
    assert made and all(o is not None for o in made)
    assert len(made) == (steps if eager else 3)      # one a forward pass whatever its layers: two to warm up and the captured one
    for a, b in zip(want, got):
        assert torch.equal(a, b)
