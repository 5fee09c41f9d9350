"""The native calls (csrc/native.cpp) against the Python path they stand in for: bit for bit on what they take, and the
Python path's own answer (conversions, broadcasts, refusals) on what they decline."""
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import _lib, layers

pytestmark = pytest.mark.gpu


class Declines:
    """Stands in for the native module: every call is the Python path's."""
    def __getattr__(self, name):
        return lambda *a: None


@pytest.fixture
def both(monkeypatch):
    def run(f):
        native = f()
        with monkeypatch.context() as m:
            m.setattr(_lib, "_native", Declines())
            m.setattr(layers, "_native", Declines())
            python = f()
        torch.cuda.synchronize()
        return native, python
    return run


def same(a, b):
    if isinstance(a, nv.Quantized):
        return same(a.weight.view(torch.int32), b.weight.view(torch.int32)) and same(a.scales, b.scales) and \
            (a.biases is None and b.biases is None or same(a.biases, b.biases))
    return a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)


def linear(n, k, quant, dtype, bias):
    q = nv.quantize(torch.randn(n, k, device="cuda").to(dtype), quant)
    return layers.QuantizedLinear(q.weight, q.scales, q.biases, torch.randn(n, device="cuda").to(dtype) if bias else None, q.quant)


QUANTS = [nv.Quant.affine(64, 4), nv.Quant.affine(32, 3), nv.Quant.new(nv.QuantMode.MXFP4), nv.Quant.new(nv.QuantMode.NVFP4)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("quant", QUANTS, ids=str)
def test_calls_equal_the_python_path(both, quant, dtype):
    torch.manual_seed(1)
    for shape in ((1, 256), (2, 3, 256), (256,), (0, 256), (70, 256)):
        for bias in (False, True):
            layer, x = linear(192, 256, quant, dtype, bias), torch.randn(shape, device="cuda").to(dtype)
            assert same(*both(lambda: layer(x))), (shape, bias)
    wide = torch.randn(4, 512, device="cuda").to(dtype)
    layer = linear(192, 256, quant, dtype, False)
    assert same(*both(lambda: layer(wide[:, ::2])))           # strided: made dense by the Python path
    mlp = layers.Mlp(linear(1024, 256, quant, dtype, False), linear(1024, 256, quant, dtype, False), linear(256, 1024, quant, dtype, True))
    fused = layers.Mlp(mlp.gate_proj, mlp.up_proj, mlp.down_proj).fuse_gate_up()
    for rows in (1, 2, 5):
        x = torch.randn(rows, 256, device="cuda").to(dtype)
        assert same(*both(lambda: mlp(x))) and same(*both(lambda: fused(x))), rows
    w = torch.randn(3, 5, 256, device="cuda").to(dtype)
    assert same(*both(lambda: nv.quantize(w, quant)))
    packed = nv.quantize(w, quant)
    for out in (None, torch.float32, torch.bfloat16):
        assert same(*both(lambda: nv.dequantize(packed, out)))
    table = nv.quantize(w.reshape(15, 256), quant)
    for ids in (torch.tensor([[3, 14], [0, 3]], device="cuda", dtype=torch.int32), torch.tensor([7], device="cuda"),
                torch.empty(0, device="cuda", dtype=torch.int32)):
        assert same(*both(lambda: nv.embedding(table, ids)))
    assert same(*both(lambda: nv.quantized_matmul(torch.ones(4, 15, device="cuda", dtype=dtype), table, transpose=False)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_attention_equals_the_python_path(both, dtype):
    torch.manual_seed(2)
    k, v = (nv.quantize(torch.randn(2, 2, 600, 64, device="cuda").to(dtype), nv.Quant.affine(32, 8)) for _ in range(2))
    q, sinks = torch.randn(2, 8, 1, 64, device="cuda").to(dtype), torch.randn(8, device="cuda").to(dtype)
    several = torch.randn(2, 8, 37, 64, device="cuda").to(dtype)
    for s in (None, sinks):
        assert same(*both(lambda: layers.quantized_attention(q, k, v, 0.125, s, causal=True)))
        assert same(*both(lambda: nv.ops.quantized_attention(q, k, v, 0.125, s)))
        for causal in (False, True):
            assert same(*both(lambda: layers.quantized_attention(several, k, v, 0.125, s, causal=causal)))


def test_refusals_are_the_python_paths():
    x = torch.randn(2, 128, device="cuda")
    q = nv.quantize(torch.randn(64, 128, device="cuda"), nv.Quant.affine(64, 4))
    with pytest.raises(nv.InvalidArgument, match="do not match"):
        nv.quantized_matmul(x[:, :64].contiguous(), q)
    with pytest.raises(nv.InvalidArgument, match="packed weights must be uint32"):
        nv.quantized_matmul(x, nv.Quantized(q.weight.view(torch.float32), q.scales, q.biases, q.quant))
    with pytest.raises(nv.InvalidArgument, match="group size 48"):
        nv.quantize(x, nv.Quant.affine(48, 4))
    mixed = nv.quantized_matmul(x.to(torch.bfloat16), q)  # promotes
    assert mixed.dtype == torch.float32


def experts(dims=256, hidden=1024, dtype=torch.bfloat16, count=8):
    """A block of experts, its gate and up projections fused."""
    put = lambda *shape: (torch.randn(shape, device="cuda") * 0.1).to(dtype)

    def projection(n, k):
        q = nv.quantize(put(count, n, k), nv.Quant.affine(64, 4))
        return layers.SwitchProjection(q.weight, q.scales, q.biases, put(count, n), q.quant)
    return layers.SwitchGlu(projection(hidden, dims), projection(hidden, dims), projection(dims, hidden)).fuse_gate_up(), put(count, dims)


@pytest.mark.parametrize("tokens", [1, 40])
def test_a_router_of_its_own(tokens):
    """`MoeMlp.route` is what routes, whoever defines it: a subclass or the block itself."""
    torch.manual_seed(4)
    glu, gate = experts()
    x = torch.randn(1, tokens, 256, device="cuda").bfloat16()
    top = torch.tensor([6, 1], dtype=torch.int32, device="cuda").expand(1, tokens, 2).contiguous()
    scores = torch.tensor([0.25, 2.0], device="cuda").bfloat16().expand(1, tokens, 2).contiguous()
    want = nv.ops.weighted_sum(glu.forward(x, top), scores)

    class Fixed(layers.MoeMlp):
        def route(self, x):
            return top, scores
    assert torch.equal(Fixed(gate, glu, 2)(x), want)
    block = layers.MoeMlp(gate, glu, 2)
    assert not torch.equal(block(x), want)
    block.route = lambda x: (top, scores)
    assert torch.equal(block(x), want)


def test_methods_of_their_own(monkeypatch):
    """A layer's method that a class or an object replaces is called, wherever the layer is held."""
    torch.manual_seed(5)
    glu, gate = experts()
    block, x = layers.MoeMlp(gate, glu, 2), torch.randn(1, 3, 256, device="cuda").bfloat16()
    plain = block(x)
    for holder, name in ((glu, "forward"), (glu.gate_up_proj, "quantized"), (glu.down_proj, "forward")):
        seen, method = [], getattr(holder, name)
        setattr(holder, name, lambda *a, **k: seen.append(1) or method(*a, **k))
        got = block(x)
        assert seen and (got.float() - plain.float()).abs().max() <= 4 * 2.0 ** -8 * plain.float().abs().max(), name
        delattr(holder, name)
        assert torch.equal(block(x), plain)
    for kind in (layers.SwitchProjection, layers.SwitchGlu):
        seen, method = [], kind.forward
        with monkeypatch.context() as m:
            m.setattr(kind, "forward", lambda *a, **k: seen.append(1) or method(*a, **k))
            block(x)
        assert seen, kind

    mlp = layers.Mlp(linear(1024, 256, nv.Quant.affine(64, 4), torch.bfloat16, True), linear(1024, 256, nv.Quant.affine(64, 4), torch.bfloat16, True),
                     linear(256, 1024, nv.Quant.affine(64, 4), torch.bfloat16, False))
    row, seen, call = x[0, :1], [], layers.QuantizedLinear.__call__
    want = mlp(row)
    with monkeypatch.context() as m:
        m.setattr(layers.QuantizedLinear, "__call__", lambda self, x: seen.append(self) or call(self, x))
        assert torch.equal(mlp(row), want) and len(seen) == 3

    table = nv.quantize(torch.randn(20, 128, device="cuda"), nv.Quant.affine(64, 4))

    class Doubled(layers.QuantizedEmbedding):
        def quantized(self):
            return nv.Quantized(self.weight, 2 * self.scales, 2 * self.biases, self.quant)
    ids = torch.tensor([3, 19], dtype=torch.int32, device="cuda")
    assert torch.equal(Doubled(table.weight, table.scales, table.biases, table.quant)(ids), 2 * nv.embedding(table, ids))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_one_query_row_alone(dtype):
    """`ops.quantized_attention` is one query row per head over caches of unsigned words: what else it refuses, so that the
    caller's masked composition runs, whatever the type, the scratch and the density."""
    k, v = (nv.quantize(torch.randn(2, 2, 96, 64, device="cuda").to(dtype), nv.Quant.affine(32, 4)) for _ in range(2))
    signed = [nv.Quantized(t.weight.view(torch.int32), t.scales, t.biases, t.quant) for t in (k, v)]
    q = torch.randn(2, 4, 3, 64, device="cuda").to(dtype)
    for scratch in (True, False):
        for queries in (q, q.transpose(1, 2).contiguous().transpose(1, 2)):
            with pytest.raises(nv.Unsupported):
                nv.ops.quantized_attention(queries, k, v, 0.125, scratch=scratch)
        with pytest.raises(nv.Unsupported):
            nv.ops.quantized_attention(q[:, :, :1].contiguous(), *signed, 0.125, scratch=scratch)
    one = q[:, :, :1].contiguous()
    composed = layers.quantized_attention(one, *signed, 0.125, fused=False)
    assert torch.equal(layers.quantized_attention(one, *signed, 0.125), composed)


def test_out_of_memory_is_torchs():
    """An allocation that fails inside a native call raises what torch's own allocation raises."""
    layer = linear(65536, 256, nv.Quant.affine(64, 4), torch.bfloat16, False)
    x = torch.randn(8192, 256, device="cuda").bfloat16()  # (an output of 1 GB)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(0.0)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            layer(x)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert layer(x).shape == (8192, 65536)


def test_streams_and_threads():
    """Calls of several host threads, each on a stream of its own: every result is the one-thread result on the default stream."""
    import threading
    torch.manual_seed(6)
    glu, gate = experts()
    moe, layer = layers.MoeMlp(gate, glu, 2), linear(1024, 256, nv.Quant.affine(64, 4), torch.bfloat16, True)
    mlp = layers.Mlp(linear(1024, 256, nv.Quant.affine(64, 4), torch.bfloat16, False), linear(1024, 256, nv.Quant.affine(64, 4), torch.bfloat16, False),
                     linear(256, 1024, nv.Quant.affine(64, 4), torch.bfloat16, False)).fuse_gate_up()
    k, v = (nv.quantize(torch.randn(1, 2, 2500, 64, device="cuda").bfloat16(), nv.Quant.affine(32, 8)) for _ in range(2))

    def work(seed):
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        put = lambda *shape: torch.randn(shape, device="cuda", generator=g).bfloat16()
        x, row, q, few = put(1, 40, 256), put(1, 256), put(1, 8, 1, 64), put(1, 8, 5, 64)
        return [moe(x), layer(x), mlp(row), mlp(x[0]), layers.quantized_attention(q, k, v, 0.125, causal=True),
                layers.quantized_attention(few, k, v, 0.125, causal=True), nv.quantize(x, nv.Quant.affine(64, 4)).weight.view(torch.int32)]
    want = [work(i) for i in range(4)]
    torch.cuda.synchronize()
    wrong = []

    def run(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                got = work(i)
                stream.synchronize()
                wrong.extend(i for a, b in zip(got, want[i]) if not torch.equal(a, b))
    threads = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("rows,dims,experts,k", [(1, 2880, 32, 4), (7, 64, 3, 3), (300, 520, 128, 8), (5, 8, 1, 1), (2, 1032, 300, 6)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_router(rows, dims, experts, k, dtype):
    """`nvq_moe_router` against float64: an unrounded probability p lies within (2 u |logit| + 3 u) p of the kernel's, u the unit
    roundoff of the type (one rounding of the logit and of the largest logit, one of p and one of the quotient; float32: the
    sums' own error, 16 u); the k chosen are the largest within twice that, in ascending order of their scores."""
    import ctypes as C
    torch.manual_seed(rows)
    x, gate = torch.randn(rows, dims, device="cuda").to(dtype), (torch.randn(experts, dims, device="cuda") * dims ** -0.5).to(dtype)
    index, scores = torch.empty(3, rows, k, dtype=torch.int32, device="cuda"), torch.empty(rows, k, dtype=dtype, device="cuda")
    nv.ops._init(x)
    p = lambda t: C.c_void_p(t.data_ptr())
    for normalize in (0, 1):
        _lib.check(_lib.load().nvq_moe_router(nv.ops._CODE[dtype], p(x), p(gate), rows, dims, experts, k, normalize, p(index[0]), p(scores),
                                              p(index[1]), p(index[2]), nv.ops._stream()))
        logits = x.double() @ gate.double().T.contiguous()
        probs = torch.softmax(logits, -1)
        u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 16 * 2.0 ** -24}[dtype]
        near = u * (2 * logits.abs().max() + 3)
        taken = torch.gather(probs, 1, index[0].long())
        assert (index[0].sort(-1).values.diff(dim=-1) > 0).all()  # distinct
        left = probs.scatter(1, index[0].long(), 0.0)
        assert (taken.min(-1).values >= left.max(-1).values * (1 - 2 * near)).all()
        assert (taken[:, 1:] >= taken[:, :-1] * (1 - 2 * near)).all()
        want = taken / taken.sum(-1, keepdim=True) if normalize else taken
        assert ((scores.double() - want).abs() <= (2 + k) * near * want + 1e-7).all()  # (the sum of k: one rounding each)
    assert torch.equal(index[1], torch.arange(rows, device="cuda", dtype=torch.int32)[:, None].expand(rows, k))
    assert torch.equal(index[2].flatten(), torch.arange(rows * k, device="cuda", dtype=torch.int32))


@pytest.mark.parametrize("experts", [1, 5, 17, 33, 64, 65])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_router_with_equal_experts(experts, dtype):
    """Equal logits in the order of a stable sort: the last experts of the highest level, then those of the one below, in ascending order."""
    import ctypes as C
    dims, rows, k = 16, 3, min(4, experts)
    x, gate = torch.ones(rows, dims, device="cuda", dtype=dtype), torch.zeros(experts, dims, device="cuda", dtype=dtype)
    gate[::16] = 0.25  # logits of 4 and 0, exact
    index, scores = torch.empty(3, rows, k, dtype=torch.int32, device="cuda"), torch.empty(rows, k, dtype=dtype, device="cuda")
    nv.ops._init(x)
    p = lambda t: C.c_void_p(t.data_ptr())
    _lib.check(_lib.load().nvq_moe_router(nv.ops._CODE[dtype], p(x), p(gate), rows, dims, experts, k, 0, p(index[0]), p(scores), p(index[1]),
                                          p(index[2]), nv.ops._stream()))
    want = sorted(range(experts), key=lambda e: (e % 16 == 0, e))[-k:]
    assert index[0].tolist() == [want] * rows


@pytest.mark.parametrize("quant", [nv.Quant.affine(64, 4), nv.Quant.affine(32, 8), nv.Quant.new(nv.QuantMode.MXFP4)], ids=str)
@pytest.mark.parametrize("dims,hidden,bias,activation", [(256, 1024, True, "swiglu_oai"), (512, 96, False, "swiglu"), (320, 640, True, "geglu")])
def test_moe_equals_the_python_path(both, quant, dims, hidden, bias, activation):
    """The same kernels but for the router's, whose logits and softmax may round the other way: each score s of a token within two of its
    steps (2 x 2^-7 s: its own and the sum's that divides it), and with it each product s y (a rounding, 2^-8, either way) and their sum."""
    torch.manual_seed(3)
    if dims % quant.group_size or hidden % quant.group_size:
        pytest.skip("not whole groups")
    put = lambda *shape: (torch.randn(shape, device="cuda") * 0.1).bfloat16()

    def projection(n, k):
        q = nv.quantize(put(8, n, k), quant)
        return layers.SwitchProjection(q.weight, q.scales, q.biases, put(8, n) if bias else None, q.quant)
    for fuse in (False, True):
        glu = layers.SwitchGlu(projection(hidden, dims), projection(hidden, dims), projection(dims, hidden), activation=activation)
        block = layers.MoeMlp(put(8, dims), glu.fuse_gate_up() if fuse else glu, 2)
        for tokens in (1, 31, 32, 200):
            x = torch.randn(1, tokens, dims, device="cuda").bfloat16()
            native, python = both(lambda: block(x))
            top, scores = block.route(x)
            terms = (scores.float()[..., None] * block.switch_mlp.forward(x, top).float()).abs().sum(-2)
            bound = (2 * 2.0 ** -7 + 2.0 ** -8) * terms + 2.0 ** -7 * python.float().abs()
            assert native.shape == python.shape and ((native.float() - python.float()).abs() <= bound).all(), (fuse, tokens)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_attention_replays_in_a_graph(dtype):
    """Captured with its workspace and replayed after other work: the eager result.  One query row on the vector kernel and on the matrix
    cores, whole and with its positions split; several rows whole, split, and in slices of the heads."""
    torch.manual_seed(7)
    for b, heads, key_heads, queries, s, d, bits in ((1, 2, 2, 1, 90, 64, 4), (1, 2, 2, 1, 5000, 128, 8), (40, 32, 4, 1, 300, 128, 4), (4, 16, 2, 1, 9000, 64, 3),
                                                     (2, 8, 2, 33, 200, 64, 4), (1, 4, 1, 3, 4000, 128, 8), (12, 8, 8, 2, 16500, 128, 4)):
        k, v = (nv.quantize(torch.randn(b, key_heads, s, d, device="cuda").to(dtype), nv.Quant.affine(32, bits)) for _ in range(2))
        q = torch.randn(b, heads, queries, d, device="cuda").to(dtype)
        run = lambda: layers.quantized_attention(q, k, v, d ** -0.5, causal=True)
        want = run()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = run()
        for _ in range(3):
            q.copy_(q.flip(0))  # (a batch of one: the same queries)
            run()
            q.copy_(q.flip(0))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want), (b, heads, queries, s)
