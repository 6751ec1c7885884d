"""GPU parity of the jagged ops against the oracle: bit-exact (pure data
movement, and one correctly rounded add per element)."""

import numpy as np
import pytest
import torch

import oracle as orc
from mx_fbgemm import bench_inputs
from tbe_helpers import gpu_us

pytestmark = pytest.mark.gpu


def _offsets(lengths):
    return bench_inputs.offsets_from_lengths(np.asarray(lengths, dtype=np.int64))


def _bits_equal(a: torch.Tensor, b: np.ndarray):
    a = a.detach().cpu().contiguous()
    if a.dtype == torch.bfloat16:
        a = a.view(torch.int16)
        b = np.asarray(b).view(np.int16)
    an = a.numpy()
    assert an.shape == b.shape, (an.shape, b.shape)
    assert an.tobytes() == np.ascontiguousarray(b).astype(an.dtype).tobytes()


CASES = [
    # (lengths, max_L, D)
    ([3, 0, 5, 1], 4, 8),          # truncation (len 5 > max_L 4) and an empty row
    ([0, 0, 0], 3, 16),            # all empty
    ([7], 7, 3),                   # odd inner size -> 4-byte path
    ([1, 2, 3, 4, 5, 6], 6, 128),  # 16-byte path
    ([2, 9, 0, 4], 3, 1),          # inner 1
]


@pytest.mark.parametrize("lengths,max_L,D", CASES)
@pytest.mark.parametrize("offset_dtype", [torch.int64, torch.int32])
def test_jagged_to_padded_dense(dev, lengths, max_L, D, offset_dtype):
    print(f"[case] j2pd lengths={lengths} max_L={max_L} D={D} {offset_dtype}", flush=True)
    rng = np.random.default_rng(1)
    off = _offsets(lengths)
    vals = rng.standard_normal((int(off[-1]), D)).astype(np.float32)
    exp = orc.jagged_to_padded_dense(vals, [off], [max_L], padding_value=-7.5)
    got = torch.ops.fbgemm.jagged_to_padded_dense(
        torch.from_numpy(vals).to(dev), [torch.from_numpy(off).to(dev, offset_dtype)], [max_L],
        -7.5)
    _bits_equal(got, exp)


@pytest.mark.parametrize("lengths,max_L,D", CASES)
def test_dense_to_jagged(dev, lengths, max_L, D):
    print(f"[case] d2j lengths={lengths} max_L={max_L} D={D}", flush=True)
    rng = np.random.default_rng(2)
    off = _offsets(lengths)
    dense = rng.standard_normal((len(lengths), max_L, D)).astype(np.float32)
    exp = orc.dense_to_jagged(dense, [off])
    got, got_off = torch.ops.fbgemm.dense_to_jagged(torch.from_numpy(dense).to(dev),
                                                     [torch.from_numpy(off).to(dev)])
    _bits_equal(got, exp)
    assert torch.equal(got_off[0].cpu(), torch.from_numpy(off))


@pytest.mark.parametrize("dtype", ["f32", "f64", "f16", "bf16"])
@pytest.mark.parametrize("lengths,max_L,D", CASES[:4])
def test_jagged_dense_add(dev, dtype, lengths, max_L, D):
    print(f"[case] add {dtype} lengths={lengths} max_L={max_L} D={D}", flush=True)
    rng = np.random.default_rng(3)
    off = _offsets(lengths)
    x = rng.standard_normal((int(off[-1]), D)).astype(np.float32)
    y = rng.standard_normal((len(lengths), max_L, D)).astype(np.float32)
    tdt = {"f32": torch.float32, "f64": torch.float64, "f16": torch.float16,
           "bf16": torch.bfloat16}[dtype]
    xt = torch.from_numpy(x).to(tdt)
    yt = torch.from_numpy(y).to(tdt)
    if dtype == "bf16":
        xn, yn = xt.view(torch.int16).numpy().view(np.uint16), yt.view(torch.int16).numpy().view(np.uint16)
    else:
        xn, yn = xt.numpy(), yt.numpy()
    exp = orc.jagged_dense_elementwise_add(xn, [off], yn, dtype)
    got, _ = torch.ops.fbgemm.jagged_dense_elementwise_add_jagged_output(
        xt.to(dev), [torch.from_numpy(off).to(dev)], yt.to(dev))
    _bits_equal(got, exp)


@pytest.mark.parametrize("dims", [1, 2, 3, 4])
@pytest.mark.parametrize("max_L,D", [(3, 4), (16, 16), (17, 16), (64, 16), (65, 16), (300, 20),
                                     (5, 3)])
def test_bag_group_sizes(dev, dims, max_L, D):
    """Chunks per innermost list either side of each group size (16, 64, 256
    threads) and past one round, 1 to 4 jagged dims, truncated and empty lists,
    values rows before the first list and past the last."""
    print(f"[case] jagged groups dims={dims} max_L={max_L} D={D}", flush=True)
    rng = np.random.default_rng(dims * 1000 + max_L + D)
    offs, maxs, n = [], [], 7
    for k in range(dims):
        top = max_L if k == dims - 1 else 3
        offs.append(_offsets(rng.integers(0, top + 3, n)))
        maxs.append(top)
        n = int(offs[-1][-1])
    vals = rng.standard_normal((n, D)).astype(np.float32)
    ot = [torch.from_numpy(o).to(dev) for o in offs]
    exp = orc.jagged_to_padded_dense(vals, offs, maxs, padding_value=2.5)
    got = torch.ops.fbgemm.jagged_to_padded_dense(torch.from_numpy(vals).to(dev), ot, maxs, 2.5)
    _bits_equal(got, exp)
    dense = rng.standard_normal(exp.shape).astype(np.float32)
    for extra in (0, 5):  # rows past the last list
        back, _ = torch.ops.fbgemm.dense_to_jagged(torch.from_numpy(dense).to(dev), ot, n + extra)
        _bits_equal(back[:n], orc.dense_to_jagged(dense, offs))
        assert not back[n:].any()
    added, _ = torch.ops.fbgemm.jagged_dense_elementwise_add_jagged_output(
        torch.from_numpy(vals).to(dev), ot, torch.from_numpy(dense).to(dev))
    _bits_equal(added, orc.jagged_dense_elementwise_add(vals, offs, dense, "f32"))


@pytest.mark.parametrize("dims", [1, 2, 3])
@pytest.mark.parametrize("head,tail", [(0, 0), (700, 0), (0, 900), (40, 30000)])
@pytest.mark.parametrize("longest,max_L,D,dt", [(50, 4, 4, "f32"), (3000, 40, 16, "f32"),
                                                (40000, 3, 5, "bf16"), (2000, 2500, 64, "bf16")])
def test_lists_past_their_cap(dev, dims, head, tail, longest, max_L, D, dt):
    """One list among 600 short ones, up to thousands of times as long: its rows
    past what its group takes (more than eight usual lists, cut by max_length or
    not) and the rows before the first list and past the last come from row
    windows of the grid, at 1 to 3 jagged dims; below and above the size at which
    a group takes any list whole.  Copy and add bit-exact."""
    print(f"[case] jagged cap dims={dims} longest={longest} max_L={max_L} D={D} head={head} "
          f"tail={tail} {dt}", flush=True)
    rng = np.random.default_rng(longest + dims)
    lengths = rng.integers(0, 5, 600)
    lengths[[0, 333, 599][dims - 1]] = longest
    outer = {1: [], 2: [[150] * 4], 3: [[2, 0, 2], [200, 50, 250, 100]]}[dims]
    maxs = {1: [], 2: [140], 3: [2, 250]}[dims] + [max_L]
    offs = [_offsets(o) for o in outer] + [_offsets(lengths) + head]
    n = int(offs[-1][-1]) + tail
    B = offs[0].size - 1
    tdt = torch.float32 if dt == "f32" else torch.bfloat16
    vals = torch.from_numpy(rng.standard_normal((n, D)).astype(np.float32)).to(tdt)
    dense = torch.from_numpy(rng.standard_normal((B, *maxs, D)).astype(np.float32)).to(tdt)
    ot = [torch.from_numpy(o).to(dev) for o in offs]
    # Expected by place: row l of list p is dense[coordinates of p, l - off[p]].
    exp = torch.zeros((n, D), dtype=tdt)
    for p in range(600):
        path, q = [], p
        for o in reversed(offs[:-1]):
            parent = int(np.searchsorted(o, q, side="right")) - 1
            path.insert(0, q - int(o[parent]))
            q = parent
        if any(c >= m for c, m in zip(path, maxs)):
            continue
        b, e = int(offs[-1][p]), int(offs[-1][p + 1])
        e = min(e, b + max_L)
        exp[b:e] = dense[(q, *path)][: e - b]
    back, _ = torch.ops.fbgemm.dense_to_jagged(dense.to(dev), ot, n)
    assert torch.equal(back.cpu().view(torch.uint8), exp.view(torch.uint8))
    added, _ = torch.ops.fbgemm.jagged_dense_elementwise_add_jagged_output(
        vals.to(dev), ot, dense.to(dev))
    want = (vals.float() + exp.float()).to(tdt)  # one rounding per element
    assert torch.equal(added.cpu().view(torch.uint8), want.view(torch.uint8))


@pytest.mark.parametrize("dims", [1, 2])
@pytest.mark.parametrize("op", ["copy", "add"])
def test_one_long_list_is_spread(dev, dims, op):
    """A batch whose rows nearly all lie in one list, or in none, takes at most ten
    times an even batch of the same rows (served by one group of threads: a
    hundred to a thousand times)."""
    print(f"[case] jagged one long list dims={dims} {op}", flush=True)
    n, L, D = 2048, 100, 16
    total = n * L

    def call(lengths, extra=0):
        offs = ([_offsets([32] * (n // 32))] if dims == 2 else []) + [_offsets(lengths)]
        maxs = [32, L] if dims == 2 else [L]
        ot = [torch.from_numpy(o).to(dev) for o in offs]
        dense = torch.randn(offs[0].size - 1, *maxs, D, device=dev)
        vals = torch.randn(int(offs[-1][-1]), D, device=dev)
        if op == "copy":
            return gpu_us(lambda: torch.ops.fbgemm.dense_to_jagged(
                dense, ot, int(offs[-1][-1]) + extra))
        return gpu_us(lambda: torch.ops.fbgemm.jagged_dense_elementwise_add_jagged_output(
            vals, ot, dense))

    even = call([L] * n)
    skewed = np.full(n, 1)
    skewed[n // 3] = total - n + 1
    one = call(skewed)
    none = call([1] * n, total - n) if op == "copy" else 0.0
    print(f"even {even:.1f} us, one list {one:.1f}, no list {none:.1f}", flush=True)
    assert one <= 10 * even and none <= 10 * even


def test_two_jagged_dims(dev):
    print("[case] j2pd/d2j two jagged dims", flush=True)
    rng = np.random.default_rng(4)
    off0 = _offsets([2, 0, 3])          # 5 level-1 rows
    off1 = _offsets([1, 4, 0, 2, 3])    # 10 values rows
    vals = rng.standard_normal((10, 6)).astype(np.float32)
    exp = orc.jagged_to_padded_dense(vals, [off0, off1], [2, 3], 0.0)
    offs = [torch.from_numpy(off0).to(dev), torch.from_numpy(off1).to(dev)]
    got = torch.ops.fbgemm.jagged_to_padded_dense(torch.from_numpy(vals).to(dev), offs, [2, 3])
    _bits_equal(got, exp)
    back = torch.ops.fbgemm.dense_to_jagged_forward(got, offs)
    _bits_equal(back, orc.dense_to_jagged(exp, [off0, off1]))


def test_config1_round_trip(dev):
    """Config 1: j2pd then d2j returns the values bit for bit (all len <= max_L)."""
    print("[case] config1 round trip B=512 D=128 max_L=64", flush=True)
    cfg = bench_inputs.config1()
    v = torch.from_numpy(cfg.values).to(dev)
    off = torch.from_numpy(cfg.offsets).to(dev)
    dense = torch.ops.fbgemm.jagged_to_padded_dense(v, [off], [cfg.max_L], 0.0)
    _bits_equal(dense, orc.jagged_to_padded_dense(cfg.values, [cfg.offsets], [cfg.max_L], 0.0))
    back, _ = torch.ops.fbgemm.dense_to_jagged(dense, [off])
    assert torch.equal(back, v)


def test_autograd(dev):
    print("[case] jagged autograd", flush=True)
    rng = np.random.default_rng(5)
    off = _offsets([2, 5, 0, 3])
    vals = torch.from_numpy(rng.standard_normal((10, 4)).astype(np.float32)).to(dev)
    vals.requires_grad_(True)
    offt = torch.from_numpy(off).to(dev)
    dense = torch.ops.fbgemm.jagged_to_padded_dense(vals, [offt], [4], 0.0)
    g = torch.from_numpy(rng.standard_normal((4, 4, 4)).astype(np.float32)).to(dev)
    (dense * g).sum().backward()
    exp = orc.dense_to_jagged(g.cpu().numpy(), [off], total_L=10)  # truncated rows get 0
    _bits_equal(vals.grad, exp)

    y = torch.from_numpy(rng.standard_normal((4, 4, 4)).astype(np.float32)).to(dev)
    y.requires_grad_(True)
    x = vals.detach().clone().requires_grad_(True)
    out, _ = torch.ops.fbgemm.jagged_dense_elementwise_add_jagged_output(x, [offt], y)
    gout = torch.from_numpy(rng.standard_normal((10, 4)).astype(np.float32)).to(dev)
    (out * gout).sum().backward()
    _bits_equal(x.grad, gout.cpu().numpy())
    _bits_equal(y.grad, orc.jagged_to_padded_dense(gout.cpu().numpy(), [off], [4], 0.0))


def test_autograd_two_jagged_dims(dev):
    """Backward of the 2-level jagged ops: d(j2pd) = d2j of the upstream
    gradient (truncated/padded positions get 0), d(d2j) = j2pd with pad 0."""
    print("[case] jagged autograd, two jagged dims", flush=True)
    rng = np.random.default_rng(6)
    off0 = _offsets([2, 0, 3])
    off1 = _offsets([1, 4, 0, 2, 3])
    offs = [torch.from_numpy(off0).to(dev), torch.from_numpy(off1).to(dev)]
    vals = torch.from_numpy(rng.standard_normal((10, 3)).astype(np.float32)).to(dev).requires_grad_()
    dense = torch.ops.fbgemm.jagged_to_padded_dense(vals, offs, [2, 3], 0.0)
    g = rng.standard_normal(tuple(dense.shape)).astype(np.float32)
    (dense * torch.from_numpy(g).to(dev)).sum().backward()
    _bits_equal(vals.grad, orc.dense_to_jagged(g, [off0, off1], total_L=10))
    d = torch.from_numpy(rng.standard_normal((3, 2, 3, 3)).astype(np.float32)).to(dev).requires_grad_()
    jv, _ = torch.ops.fbgemm.dense_to_jagged(d, offs)
    gj = rng.standard_normal(tuple(jv.shape)).astype(np.float32)
    (jv * torch.from_numpy(gj).to(dev)).sum().backward()
    _bits_equal(d.grad, orc.jagged_to_padded_dense(gj, [off0, off1], [2, 3], 0.0))


def test_jagged_to_padded_dense_backward_op(dev):
    print("[case] jagged_to_padded_dense_backward op", flush=True)
    rng = np.random.default_rng(8)
    off = _offsets([3, 0, 6, 2])
    g = rng.standard_normal((4, 4, 5)).astype(np.float32)
    got = torch.ops.fbgemm.jagged_to_padded_dense_backward(
        torch.from_numpy(g).to(dev), [torch.from_numpy(off).to(dev)], 11)
    _bits_equal(got, orc.dense_to_jagged(g, [off], total_L=11))


@pytest.mark.parametrize("dtype", ["f32", "f64", "f16", "bf16"])
@pytest.mark.parametrize("lengths,max_L,D", CASES)
def test_jagged_dense_mul(dev, dtype, lengths, max_L, D):
    """x * y at the jagged coordinates (x * 0 past max_L), bit for bit."""
    print(f"[case] mul {dtype} lengths={lengths} max_L={max_L} D={D}", flush=True)
    rng = np.random.default_rng(13)
    off = _offsets(lengths)
    tdt = {"f32": torch.float32, "f64": torch.float64, "f16": torch.float16,
           "bf16": torch.bfloat16}[dtype]
    xt = torch.from_numpy(rng.standard_normal((int(off[-1]), D))).to(tdt)
    yt = torch.from_numpy(rng.standard_normal((len(lengths), max_L, D))).to(tdt)
    if dtype == "bf16":
        xn, yn = xt.view(torch.int16).numpy().view(np.uint16), yt.view(torch.int16).numpy().view(np.uint16)
    else:
        xn, yn = xt.numpy(), yt.numpy()
    exp = orc.jagged_dense_elementwise_mul(xn, [off], yn, dtype)
    got = torch.ops.fbgemm.jagged_dense_elementwise_mul(xt.to(dev), [torch.from_numpy(off).to(dev)],
                                                        yt.to(dev))
    _bits_equal(got, exp)


def test_jagged_dense_mul_two_dims_and_autograd(dev):
    """Two jagged dims; d/dx = grad * y at the coordinates, d/dy = the padded
    dense of grad * x, both against the oracle's gather / scatter, bit for bit."""
    print("[case] mul two jagged dims + autograd", flush=True)
    rng = np.random.default_rng(14)
    off0 = _offsets([2, 0, 3])
    off1 = _offsets([1, 4, 0, 2, 3])
    offs = [torch.from_numpy(off0).to(dev), torch.from_numpy(off1).to(dev)]
    x = rng.standard_normal((10, 3)).astype(np.float32)
    y = rng.standard_normal((3, 2, 3, 3)).astype(np.float32)
    xt = torch.from_numpy(x).to(dev).requires_grad_()
    yt = torch.from_numpy(y).to(dev).requires_grad_()
    out = torch.ops.fbgemm.jagged_dense_elementwise_mul(xt, offs, yt)
    _bits_equal(out, orc.jagged_dense_elementwise_mul(x, [off0, off1], y, "f32"))
    g = rng.standard_normal((10, 3)).astype(np.float32)
    (out * torch.from_numpy(g).to(dev)).sum().backward()
    _bits_equal(xt.grad, orc.jagged_dense_elementwise_mul(g, [off0, off1], y, "f32"))
    _bits_equal(yt.grad, orc.jagged_to_padded_dense((g * x).astype(np.float32), [off0, off1],
                                                    [2, 3], 0.0))


@pytest.mark.parametrize("lengths,max_L,D", CASES)
def test_jagged_2d_to_dense(dev, lengths, max_L, D):
    print(f"[case] jagged_2d_to_dense lengths={lengths} max_L={max_L} D={D}", flush=True)
    rng = np.random.default_rng(15)
    off = _offsets(lengths)
    v = rng.standard_normal((int(off[-1]), D)).astype(np.float32)
    vt = torch.from_numpy(v).to(dev).requires_grad_()
    got = torch.ops.fbgemm.jagged_2d_to_dense(vt, torch.from_numpy(off).to(dev), max_L)
    _bits_equal(got, orc.jagged_to_padded_dense(v, [off], [max_L], 0.0))
    g = rng.standard_normal(tuple(got.shape)).astype(np.float32)
    (got * torch.from_numpy(g).to(dev)).sum().backward()
    _bits_equal(vt.grad, orc.dense_to_jagged(g, [off], total_L=int(off[-1])))


@pytest.mark.parametrize("dtype,pad", [(np.int64, -1), (np.int64, (1 << 62) + 3),
                                       (np.int32, 7), (np.float32, -2)])
def test_jagged_1d_to_dense(dev, dtype, pad):
    """Integer padding keeps every bit of an int64 (2^62 + 3 is not a double)."""
    print(f"[case] jagged_1d_to_dense {np.dtype(dtype).name} pad={pad}", flush=True)
    rng = np.random.default_rng(16)
    lengths = [3, 0, 6, 1, 2]
    off = _offsets(lengths)
    v = rng.integers(-1000, 1000, int(off[-1])).astype(dtype)
    got = torch.ops.fbgemm.jagged_1d_to_dense(torch.from_numpy(v).to(dev),
                                              torch.from_numpy(off).to(dev), 4, pad)
    exp = np.full((len(lengths), 4), pad, dtype)
    for b, n in enumerate(lengths):
        k = min(n, 4)
        exp[b, :k] = v[off[b]:off[b] + k]
    _bits_equal(got, exp)


def test_jagged_dense_add_autograd_two_dims(dev):
    """The add's backward with two jagged dims: grad_x = grad, grad_y = the
    padded dense of grad (the offsets list is one argument of the node)."""
    print("[case] add autograd two jagged dims", flush=True)
    rng = np.random.default_rng(17)
    off0 = _offsets([2, 0, 3])
    off1 = _offsets([1, 4, 0, 2, 3])
    offs = [torch.from_numpy(off0).to(dev), torch.from_numpy(off1).to(dev)]
    xt = torch.from_numpy(rng.standard_normal((10, 3)).astype(np.float32)).to(dev).requires_grad_()
    yt = torch.from_numpy(rng.standard_normal((3, 2, 3, 3)).astype(np.float32)).to(dev).requires_grad_()
    out, _ = torch.ops.fbgemm.jagged_dense_elementwise_add_jagged_output(xt, offs, yt)
    g = rng.standard_normal((10, 3)).astype(np.float32)
    (out * torch.from_numpy(g).to(dev)).sum().backward()
    _bits_equal(xt.grad, g)
    _bits_equal(yt.grad, orc.jagged_to_padded_dense(g, [off0, off1], [2, 3], 0.0))
