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
