"""Weight tiles whose k blocks begin with another one each (rows a multiple of 8192 bytes apart; experts: 4096): the products against 64 bits.

Sums of K products of |a| <= 1 stored in bf16: the result's rounding (2^-9 relative) and the 32-bit sums' error (K 2^-24 of the sum of
magnitudes, far below it) allow 2^-8 of the row's scale."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _draw(*shape, g, dtype=torch.bfloat16):
    return (torch.rand(*shape, generator=g, device=DEV) * 2 - 1).to(dtype)


def _close(got, want):
    scale = want.norm() / want.numel() ** 0.5
    err = (got.double() - want).abs()
    assert (err / (want.abs() + scale)).max() < 2 ** -8


# one slice and fewer or more tiles than blocks, slices that begin 4096 bytes apart and others, 8 to 128 rows and 129 to 256, two row blocks, a
# hanging last tile
@pytest.mark.parametrize("n,k", [(33056, 4096), (24576, 4096), (15360, 4096), (10368, 4096), (4112, 4096), (4096, 8192), (2048, 16384), (4096, 12288)])
@pytest.mark.parametrize("m", [1, 33, 64, 128, 200, 300])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear(n, k, m, dtype):
    from vllm_omni_amd import ops

    g = torch.Generator(device=DEV).manual_seed(n + m)
    x, w, b = _draw(m, k, g=g, dtype=dtype), _draw(n, k, g=g, dtype=dtype), _draw(n, g=g, dtype=dtype)
    cols = torch.randint(0, n, (257,), generator=g, device=DEV)
    cols[:2] = torch.tensor([0, n - 1])
    want = x.double() @ w[cols].double().t()
    _close(ops.linear(x, w, b)[:, cols], want + b[cols].double())
    if n % 32 == 0:      # gate and up rows of the same columns
        i = n // 2
        c = cols % i
        gate, up = ((x.double() @ w[c + o].double().t()).to(dtype).double() for o in (0, i))
        got = ops.linear_silu_mul(x, w)[:, c].double()
        ref = torch.nn.functional.silu(gate) * up
        # the two 16-bit roundings in front: each half an ulp of its factor
        scale = ref.norm() / ref.numel() ** 0.5
        assert ((got - ref).norm() / ref.norm()) < 2 ** -7 and ((got - ref).abs() / (ref.abs() + scale)).max() < 2 ** -5


@pytest.mark.parametrize("h,i,e,top,t", [(4096, 1536, 8, 2, 3), (4096, 256, 16, 4, 60), (2048, 512, 16, 4, 150), (4096, 1536, 64, 8, 64), (4096, 1536, 64, 8, 200),
                                         (2048, 768, 64, 8, 200), (8192, 128, 8, 2, 40), (2048, 2048, 8, 2, 40)])
@pytest.mark.parametrize("act", ["silu_gated", "relu_squared"])
def test_experts(h, i, e, top, t, act, monkeypatch):
    from vllm_omni_amd import ops

    g = torch.Generator(device=DEV).manual_seed(h + t)
    ups = 2 if act == "silu_gated" else 1
    x = _draw(t, h, g=g)
    wu, wd = _draw(e, ups * i, h, g=g) * h ** -0.5, _draw(e, h, i, g=g) * i ** -0.5
    ids = torch.rand(t, e, generator=g, device=DEV).argsort(-1)[:, :top].int().contiguous()
    pw = torch.rand(t, top, generator=g, device=DEV)
    pick = torch.randint(0, t, (min(t, 12),), generator=g, device=DEV)
    want = []
    for tok in pick.tolist():
        for j in range(top):
            u = x[tok].double() @ wu[ids[tok, j]].double().t()
            mid = torch.nn.functional.silu(u[:i]) * u[i:] if ups == 2 else torch.relu(u) ** 2
            want.append(mid @ wd[ids[tok, j]].double().t())
    want = torch.stack(want)
    for mode in (None, "always"):
        if mode:
            monkeypatch.setenv("MI_MOE_GEMM", mode)
        r = ops.moe_expert_rows(x, ids, pw, wu, wd, act)
        rows = r.row_of_pair.view(t, top)[pick].reshape(-1).long()
        got = r.part[rows].double()
        # activations are stored in bf16 in front of the second product
        assert (got - want).norm() / want.norm() < 2 ** -7


# where gated tiles of under 64 columns begin to be turned, and end: 209 to 249 tiles of K 4096 to 64 rows, longer K to 128 and 224
@pytest.mark.parametrize("inter,k,rows", [(6656, 4096, (64,)), (6688, 4096, (33, 64, 65)), (7968, 4096, (1, 64)), (8000, 4096, (64,)), (3584, 4096, (32, 65)), (4096, 8192, (128, 224, 225)), (2048, 12288, (16, 128, 129))])
def test_gated_lines(inter, k, rows):
    from vllm_omni_amd import ops

    g = torch.Generator(device=DEV).manual_seed(inter + k)
    w = _draw(2 * inter, k, g=g)
    c = torch.randint(0, inter, (257,), generator=g, device=DEV)
    for m in rows:
        x = _draw(m, k, g=g)
        gate, up = ((x.double() @ w[c + o].double().t()).to(w.dtype).double() for o in (0, inter))
        ref, got = torch.nn.functional.silu(gate) * up, ops.linear_silu_mul(x, w)[:, c].double()
        scale = ref.norm() / ref.numel() ** 0.5      # (as in test_linear)
        assert ((got - ref).norm() / ref.norm()) < 2 ** -7 and ((got - ref).abs() / (ref.abs() + scale)).max() < 2 ** -5


# 32-bit slabs and the launches behind them: the bits of the linear, and the squared relu's sums
@pytest.mark.parametrize("n,k", [(15360, 4096), (8192, 8192), (4096, 16384)])
@pytest.mark.parametrize("m", [1, 64, 128, 200])
def test_slabs(n, k, m):
    from vllm_omni_amd import ops

    g = torch.Generator(device=DEV).manual_seed(n + m)
    x, w, b = _draw(m, k, g=g), _draw(n, k, g=g), _draw(n, g=g)
    part = ops.linear_partials(x, w, b)
    got = part.materialize()
    assert torch.equal(got, ops.linear(x, w, b))
    cols = torch.randint(0, n, (257,), generator=g, device=DEV)
    want = x.double() @ w[cols].double().t()
    _close(got[:, cols], want + b[cols].double())
    _close(ops.linear_relu_squared(x, w)[:, cols], torch.relu(want) ** 2)


# int8: K counts pairs of bytes, so rows of 8192 and 16384 bytes are turned; integer sums have one value whatever their order
@pytest.mark.parametrize("n,k", [(33056, 8192), (10368, 8192), (4112, 8192), (4096, 16384)])
@pytest.mark.parametrize("m", [1, 64, 128, 200, 300])
def test_int8(n, k, m):
    from vllm_omni_amd import ops

    g = torch.Generator(device=DEV).manual_seed(n + m)
    xq, wq = (torch.randint(-128, 128, s, generator=g, device=DEV, dtype=torch.int32).to(torch.int8) for s in ((m, k), (n, k)))
    xs, ws = torch.rand(m, generator=g, device=DEV) * 0.05 + 1e-3, torch.rand(n, generator=g, device=DEV) * 0.01 + 1e-4
    b = _draw(n, g=g)
    got = ops.int8_linear_q(xq, xs, wq, ws, b, torch.bfloat16)
    assert torch.equal(got, ops.int8_gemm_dequant(xq, xs, wq, ws, b, torch.bfloat16))
    cols = torch.randint(0, n, (129,), generator=g, device=DEV)
    want = (xq.double() @ wq[cols].double().t()) * xs[:, None].double() * ws[cols].double() + b[cols].double()
    _close(got[:, cols], want)


@pytest.mark.parametrize("inter,k,m", [(16528, 8192, 1), (16528, 8192, 64), (12288, 8192, 200), (5184, 16384, 128), (2048, 8192, 300)])
def test_int8_gated(inter, k, m):
    from vllm_omni_amd import ops

    g = torch.Generator(device=DEV).manual_seed(inter + m)
    x = _draw(m, k, g=g)
    wq, ws = ops.dynamic_int8_quant(_draw(2 * inter, k, g=g) * 0.05)
    gt, up = ops.int8_gemm_dequant(*ops.dynamic_int8_quant(x), wq, ws, None, torch.bfloat16).float().split(inter, -1)
    want, got = torch.nn.functional.silu(gt) * up, ops.int8_linear_silu_mul(x, wq, ws).float()
    # both round the two integer products to 16 bits first: one more rounding, and the error of the fast exponential (far below it)
    assert ((got - want).abs() <= want.abs() * 2.0 ** -7 + 1e-6).all()


# every row by itself: rounding of the gate, the activations and the results is about 2^-8 of a row's norm
@pytest.mark.parametrize("h,i,e,top,t", [(4096, 1536, 64, 8, 64), (4096, 1536, 64, 8, 200), (2048, 768, 64, 8, 200), (4096, 256, 16, 4, 60), (4096, 512, 8, 4, 700)])
@pytest.mark.parametrize("act", ["silu_gated", "relu_squared"])
def test_every_row_of_the_experts(h, i, e, top, t, act):
    from vllm_omni_amd import ops

    g = torch.Generator(device=DEV).manual_seed(h + t)
    ups = 2 if act == "silu_gated" else 1
    x = _draw(t, h, g=g)
    wu, wd = _draw(e, ups * i, h, g=g) * h ** -0.5, _draw(e, h, i, g=g) * i ** -0.5
    ids = torch.rand(t, e, generator=g, device=DEV).argsort(-1)[:, :top].int().contiguous()
    r = ops.moe_expert_rows(x, ids, torch.rand(t, top, generator=g, device=DEV), wu, wd, act)
    got = r.part[r.row_of_pair.long()].view(t, top, h).double()
    for j in range(e):
        tok, place = (ids == j).nonzero(as_tuple=True)
        u = x[tok].double() @ wu[j].double().t()
        mid = torch.nn.functional.silu(u[:, :i]) * u[:, i:] if ups == 2 else torch.relu(u) ** 2
        want = mid @ wd[j].double().t()
        assert ((got[tok, place] - want).norm(dim=-1) <= want.norm(dim=-1) * 2 ** -7).all(), j
