"""Which weights the layers hand to the kernels (host logic only: the kernel calls are recorded)."""

import pytest
import torch

from looped_blockell import kernels


@pytest.fixture
def looped(monkeypatch):
    """A CPU LoopedSwiGLU and the (gate, up, down) values that each of its calls passed to a kernel."""
    from looped_blockell.layers import LoopedSwiGLU
    seen = []

    def looped_bias(h, scale, vg, cg, bg, vu, cu, bu, vd, cd, bd, L, eps=1e-5):
        seen.append((vg, vu, vd))
        return h * vg.flatten()[0]

    monkeypatch.setattr(kernels, "looped_swiglu_bias", looped_bias)
    return LoopedSwiGLU(64, 128, 2, tile_size=16, density=0.5), seen


def test_looped_forward_reads_the_weights_of_the_call(looped):
    """A gradient-free looped forward rounds the weights as they are at the call, whether or not the write
    before it raised a version (a captured call then holds the rounding, and replays follow the weights)."""
    m, seen = looped
    h = torch.zeros(3, 64, dtype=torch.bfloat16)
    with torch.no_grad():
        m(h)
        for write in (lambda p: p.data.mul_(2), lambda p: p.data.copy_(torch.randn(p.shape)), lambda p: p.mul_(3)):
            for lin in (m.mlp.w_gate, m.mlp.w_up, m.mlp.w_down):
                write(lin.values)
            m(h)
            for got, lin in zip(seen[-1], (m.mlp.w_gate, m.mlp.w_up, m.mlp.w_down)):
                assert torch.equal(got, lin.values.detach().to(torch.bfloat16))
    assert m.mlp._frozen is None          # no copy outlives the call


def test_looped_forward_under_vmap_over_weights(looped):
    m, _ = looped
    gates = torch.randn(2, *m.mlp.w_gate.values.shape)
    h = torch.ones(3, 64, dtype=torch.bfloat16)
    with torch.no_grad():
        out = torch.func.vmap(lambda v: torch.func.functional_call(m, {"mlp.w_gate.values": v}, (h,)))(gates)
    assert torch.equal(out[:, 0, 0], gates.flatten(1)[:, 0].to(torch.bfloat16))


@pytest.mark.gpu
@pytest.mark.parametrize("N", [5, 130])
@pytest.mark.parametrize("tile", [16, 64])
def test_captured_looped_forward_follows_its_weights(gpu, N, tile):
    """Replays of a captured gradient-free looped forward use the weights of the moment, with eager
    forwards (which must not disturb what the graph reads) and weight writes between them."""
    from looped_blockell.layers import LoopedSwiGLU
    torch.manual_seed(4)

    def make():
        return LoopedSwiGLU(256, 512, 3, tile_size=tile, density=0.5, device="cuda")

    m, x = make(), torch.randn(N, 256, device="cuda").to(torch.bfloat16)

    def fresh():
        n = make()
        n.load_state_dict(m.state_dict())
        return n(x)

    with torch.no_grad():
        m(x)
        for p in m.parameters():
            p.mul_(1.5)                       # the first forward after this write is the captured one
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            y = m(x)
        assert torch.equal(m(x), fresh())
        last = None
        for k in range(4):
            for lin in (m.mlp.w_gate, m.mlp.w_up, m.mlp.w_down):
                w = torch.randn_like(lin.values) * 0.05
                if k % 2:
                    lin.values.data.copy_(w)
                else:
                    lin.values.copy_(w)
            if k >= 2:
                assert torch.equal(m(x), fresh())
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, fresh()), k
            assert last is None or not torch.equal(y, last)
            last = y.clone()


@pytest.mark.gpu
def test_looped_forward_on_two_streams(gpu):
    """A forward on another stream right after a weight write on that stream sees the written weights."""
    from looped_blockell.layers import LoopedSwiGLU
    torch.manual_seed(5)
    m = LoopedSwiGLU(256, 512, 2, tile_size=16, density=0.5, device="cuda")
    x = torch.randn(70, 256, device="cuda").to(torch.bfloat16)
    s = torch.cuda.Stream()
    with torch.no_grad():
        m(x)
        for _ in range(3):
            s.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(s):
                m.mlp.w_gate.values.mul_(1.25)
                a = m(x)
            torch.cuda.current_stream().wait_stream(s)
            assert torch.equal(a, m(x))


def _recorded_training(monkeypatch):
    """Record the calls that MLPBlock makes for a forward with gradients (CPU stand-ins)."""
    calls = []
    monkeypatch.setattr(kernels, "swiglu_train", lambda x, vg, *a, **k: calls.append(("train", vg, a, k)) or x * 1.0)
    monkeypatch.setattr(kernels, "swiglu", lambda x, vg, *a, **k: calls.append(("bf16", vg, a, k)) or x * 1.0)
    monkeypatch.setattr(kernels, "looped_swiglu_train",
                        lambda h, s, vg, *a, **k: calls.append(("looped", vg, a, k)) or h * 1.0)
    return calls


@pytest.mark.parametrize("where", ["subclass", "instance"])
def test_training_forward_uses_an_overridden_swiglu_weights(monkeypatch, where):
    """A replaced ``swiglu_weights`` (a fake quantiser, say) decides the weights of a training forward."""
    from looped_blockell.layers import LoopedSwiGLU, MLPBlock
    from looped_blockell.layers import norms
    calls = _recorded_training(monkeypatch)

    def doubled(self):
        w = MLPBlock.swiglu_weights(self)
        return (2 * w[0], *w[1:])

    class Doubled(MLPBlock):
        swiglu_weights = doubled

    kw = dict(use_swiglu=True, tile_size=16, density=0.5)
    if where == "subclass":
        m = Doubled(64, 128, **kw)
    else:
        m = MLPBlock(64, 128, **kw)
        m.swiglu_weights = lambda: doubled(m)
    m(torch.zeros(3, 64, dtype=torch.bfloat16))
    assert calls[-1][0] == "bf16" and torch.equal(calls[-1][1], 2 * m.w_gate.values.to(torch.bfloat16))
    monkeypatch.setattr(norms.RMSNorm, "forward", lambda self, x: x)
    loop = LoopedSwiGLU(64, 128, 2, tile_size=16, density=0.5)
    loop.mlp = m
    loop(torch.zeros(3, 64, dtype=torch.bfloat16))
    assert calls[-1][0] == "bf16" and torch.equal(calls[-1][1], 2 * m.w_gate.values.to(torch.bfloat16))


def test_ternary_forward_uses_an_overridden_prepared(monkeypatch):
    """A replaced ``prepared`` decides the weights of a ternary forward."""
    from looped_blockell.layers import TernaryBlockELLWeight, TernaryMLPBlock
    seen = []
    monkeypatch.setattr(kernels, "quantize_act_int8", lambda x: (x, x))
    monkeypatch.setattr(kernels, "ternary_prepare", lambda *t: "built")
    monkeypatch.setattr(kernels, "ternary_swiglu_fwd_prepared", lambda xq, sx, prep, *a: seen.append(prep) or xq)

    def weight(R, K):
        return TernaryBlockELLWeight(torch.zeros(R, K, 16, 1, dtype=torch.int32), torch.ones(R, K),
                                     torch.zeros(R, K, dtype=torch.int32))

    class Own(TernaryMLPBlock):
        def prepared(self):
            return "own"

    x = torch.zeros(3, 32)
    for cls, want in ((TernaryMLPBlock, "built"), (Own, "own")):
        cls(weight(4, 1), weight(4, 1), weight(2, 1))(x)
        assert seen[-1] == want


def test_looped_training_with_another_mlp(monkeypatch):
    """A looped block whose MLP was replaced by a GELU one trains through that module's own calls."""
    from looped_blockell.layers import LoopedSwiGLU, MLPBlock, norms
    _recorded_training(monkeypatch)
    monkeypatch.setattr(norms.RMSNorm, "forward", lambda self, x: x)
    monkeypatch.setattr(MLPBlock, "_gelu", lambda self, x: x + 1)
    loop = LoopedSwiGLU(64, 128, 3, tile_size=16, density=0.5)
    loop.mlp = MLPBlock(64, 128, tile_size=16)
    out = loop(torch.ones(3, 64, dtype=torch.bfloat16))
    assert (out == 15).all()                  # h <- h + (h + 1), three times from 1
