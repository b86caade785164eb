"""What the layer calls (``ffn.ffn_forward`` / ``ffn_backward``, and the operators in front of them) do with arguments that
do not fit: converted where that is exact, refused where the kernels would read something else than the tensor."""
import dataclasses
import types
import weakref

import pytest
import torch

from analog_moe_amd import _abi, ffn
from tests import util
from tests.test_emu_kernels import emu_ops  # noqa: F401  (the host build behind analog_moe_amd.ops)

E, D, F, T, K = 3, 32, 24, 10, 2


def problem(dtype=torch.float32, **kw):
    pr = util.make_problem(7, **{**dict(T=T, D=D, E=E, F=F, k=K, dtype=dtype), **kw})
    pr["ir"] = torch.linspace(1.0, 2.0, 2 * E).reshape(2, E, 1)
    return pr


def forward(pr, cfg, **swap):
    a = {**pr, **swap}
    return ffn.ffn_forward(a["x"], a["keys"], a["values"], a["ir"], a["gate"], a["idx"], cfg)


def backward(pr, cfg, saved, want_ir_grad=True, ir_dtype=torch.float32, **swap):
    a = {**pr, **dict(zip(("p1", "z", "perm", "in_index", "offsets", "z_scale", "ir_up", "ir_dn"), saved[1:])), **swap}
    return ffn.ffn_backward(a["dy"], a["x"], a["keys"], a["values"], a["gate"], a["idx"], a["p1"], a["z"], a["z_scale"],
                            a["perm"], a["in_index"], a["offsets"], a["ir_up"], a["ir_dn"], cfg, want_ir_grad, ir_dtype)


def same(a, b):
    return all((p is None and q is None) or torch.equal(p, q) for p, q in zip(a, b))


PLAIN = ffn.FFNConfig(inp_res=1 / 127)
ADC = dataclasses.replace(PLAIN, out_bound=12.0, out_res=254.0)


def test_input_range_of_another_type(emu_ops):
    pr = problem()
    want = forward(pr, PLAIN)
    got = forward(pr, PLAIN, ir=pr["ir"].double())
    assert same(got, want)
    with pytest.raises(TypeError):              # the tables' launch reads the parameter itself
        forward(pr, ADC, ir=pr["ir"].double())
    with pytest.raises(TypeError):              # and the per-expert sums are written in its type
        backward(pr, PLAIN, got, ir_dtype=torch.float64)
    assert backward(pr, PLAIN, got, want_ir_grad=False, ir_dtype=torch.float64)[3] is None


@pytest.mark.parametrize("cfg", [PLAIN, ADC], ids=["plain", "adc"])
def test_input_range_that_is_no_table_of_both_projections(emu_ops, cfg):
    pr = problem()
    with pytest.raises((RuntimeError, ValueError)):
        forward(pr, cfg, ir=torch.ones(2 * E + 1))
    with pytest.raises((RuntimeError, ValueError)):            # fewer columns than K-tiles
        forward(pr, dataclasses.replace(cfg, bounds_up=(0, 16, D)))


def injected(pr, dtype=torch.float32, nt=1):
    g = torch.Generator().manual_seed(3)
    return dict(noise_std=0.04, noise_up=(0.1 * torch.randn(nt, T * K, F, generator=g)).to(dtype),
                noise_down=(0.1 * torch.randn(1, T * K, D, generator=g)).to(dtype))


def test_injected_noise_of_another_type_or_layout(emu_ops):
    pr = problem()
    noise = injected(pr, torch.bfloat16)
    want = forward(pr, dataclasses.replace(ADC, **{n: t.float() if n != "noise_std" else t for n, t in noise.items()}))
    assert same(forward(pr, dataclasses.replace(ADC, **noise)), want)
    turned = noise["noise_up"].float().transpose(1, 2).contiguous().transpose(1, 2)
    assert not turned.is_contiguous() and same(forward(pr, dataclasses.replace(ADC, **{**noise, "noise_up": turned})), want)


@pytest.mark.parametrize("which", ["noise_up", "noise_down"])
def test_injected_noise_of_another_size(emu_ops, which):
    pr = problem()
    noise = injected(pr)
    noise[which] = noise[which][:, 1:].contiguous()
    with pytest.raises(ValueError):
        forward(pr, dataclasses.replace(ADC, **noise))


@pytest.mark.parametrize("per_channel", [False, True])
def test_max_w_tables_say_their_own_columns(emu_ops, per_channel):
    """[E] (or [E, 1]) and [E, N] tables of the caller, whatever noise_per_channel says of tables made here, one of each
    kind among them, in any floating type; the down-projection's alone is not used."""
    pr = problem()
    cfg = dataclasses.replace(ADC, noise_std=0.04, noise_seed=5)
    up, dn = (torch.rand(E, n, generator=torch.Generator().manual_seed(n)) + 1.0 for n in (F, D))
    one_up, one_dn = up[:, :1].clone(), dn[:, :1].clone()

    def run(u, d, pc=per_channel):
        return forward(pr, dataclasses.replace(cfg, wmax_up=u, wmax_down=d, noise_per_channel=pc))
    wide = run(up, dn, True)
    narrow = run(one_up, one_dn, False)
    assert same(run(up, dn), wide) and same(run(one_up, one_dn), narrow)
    assert same(run(one_up[:, 0], one_dn[:, 0]), narrow)
    assert same(run(one_up, dn)[1:2], narrow[1:2]) and same(run(up, one_dn)[1:2], wide[1:2])
    assert same(run(one_up.expand(E, F), dn), run(one_up, dn))
    assert same(run(up.double(), dn.double()), wide)
    assert same(run(None, one_dn), forward(pr, dataclasses.replace(cfg, noise_per_channel=per_channel)))
    for bad in ((up[:, :-1], dn), (up, dn[:, 1:])):
        with pytest.raises((ValueError, _abi.AmoeError)):
            run(*bad)
    assert same(forward(pr, dataclasses.replace(PLAIN, wmax_up=up[:, :5], wmax_down=dn)), forward(pr, PLAIN))   # no reader


def test_late_max_w_table_is_converted_after_its_event(emu_ops, monkeypatch):
    """A table of the down-projection that another stream still makes: what converts it waits for its event first."""
    pr, order = problem(), []
    event = type("Event", (), {"cuda_event": 0})()
    stream = type("Stream", (), {"wait_event": lambda self, e: order.append(e)})()
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: stream)
    cfg = dataclasses.replace(ADC, wmax_up=torch.ones(E, 1), wmax_down=torch.ones(E, 1), down_ready=event)
    forward(pr, cfg)
    assert order == []                                         # (the library's own launch waits)
    forward(pr, dataclasses.replace(cfg, wmax_down=cfg.wmax_down.double()))
    forward(pr, dataclasses.replace(cfg, wmax_up=torch.ones(E, F)))
    assert order == [event, event]


@pytest.mark.parametrize("word", [torch.zeros(1, dtype=torch.int32), torch.zeros(2, dtype=torch.int64), torch.zeros(1)])
def test_seed_word_that_is_none(emu_ops, word):
    pr = problem()
    with pytest.raises(ValueError):
        forward(pr, dataclasses.replace(ADC, noise_std=0.04, noise_seed_dev=word))
    with pytest.raises(ValueError):
        forward(pr, dataclasses.replace(PLAIN, noise_seed_dev=word))


def test_backward_of_another_gradient(emu_ops):
    pr = problem()
    saved = forward(pr, ADC)
    want = backward(pr, ADC, saved)
    assert same(backward(pr, ADC, saved, dy=pr["dy"].reshape(2, T // 2, D)), want)
    assert same(backward(pr, ADC, saved, dy=pr["dy"].t().contiguous().t()), want)
    for bad in (pr["dy"][1:], pr["dy"][:, 1:], torch.cat((pr["dy"], pr["dy"]))):
        with pytest.raises((ValueError, RuntimeError)):
            backward(pr, ADC, saved, dy=bad)
    with pytest.raises(TypeError):
        backward(pr, ADC, saved, dy=pr["dy"].double())


def test_backward_of_other_saved_tensors(emu_ops):
    """Hooks on saved tensors, and callers of the operators, may hand over copies in another layout, or anything."""
    pr = problem()
    saved = forward(pr, ADC)
    want = backward(pr, ADC, saved)
    y, p1, z, perm, in_index, offsets, z_scale, ir_up, ir_dn = saved

    def turned(t):
        return t.t().contiguous().t()
    assert same(backward(pr, ADC, saved, p1=turned(p1), z=turned(z), idx=turned(pr["idx"]), gate=turned(pr["gate"]),
                         ir_up=ir_up.double(), ir_dn=ir_dn.double()), want)
    wrong = [dict(p1=p1[1:]), dict(z=z[1:]), dict(z=z[:, 1:]), dict(perm=perm[1:]), dict(in_index=in_index[1:]),
             dict(offsets=offsets[1:]), dict(perm=perm.long()), dict(in_index=in_index.float()), dict(offsets=offsets.long()),
             dict(ir_up=ir_up[1:]), dict(ir_dn=torch.ones(E, 3)), dict(idx=pr["idx"][1:]), dict(gate=pr["gate"][1:]), dict(p1=p1.double()),
             dict(z=z.double()), dict(z=z.to(torch.uint8)), dict(perm=torch.stack((perm, perm), 1)[:, 0])]
    for swap in wrong:
        with pytest.raises((ValueError, TypeError)):
            backward(pr, ADC, saved, **swap)


def test_every_tensor_must_lie_on_the_gpu(emu_ops, monkeypatch):
    """A pointer to host memory in a kernel is a fault on the GPU: every tensor of a call passes the device check."""
    pr = problem()
    noise = injected(pr)
    cfg = dataclasses.replace(ADC, **noise, wmax_up=torch.ones(E, 1), wmax_down=torch.ones(E, 1), noise_seed_dev=torch.zeros(1, dtype=torch.int64))
    saved = forward(pr, cfg)
    seen = []
    monkeypatch.setattr(emu_ops, "_need_gpu", lambda *t: seen.extend(id(v) for v in t))
    forward(pr, cfg)
    for t in (*(pr[n] for n in ("x", "keys", "values", "ir", "gate", "idx")), cfg.noise_up, cfg.noise_down, cfg.wmax_up, cfg.wmax_down,
              cfg.noise_seed_dev):
        assert id(t) in seen
    del seen[:]
    backward(pr, cfg, saved)
    for t in (*(pr[n] for n in ("dy", "x", "keys", "values", "gate", "idx")), *(t for t in saved[1:])):
        assert id(t) in seen


def test_heads_of_gate_and_ids_agree(emu_ops):
    pr = problem()
    want = forward(pr, PLAIN)
    lead = dict(gate=pr["gate"].reshape(2, T // 2, K), idx=pr["idx"].reshape(2, T // 2, K))
    assert same(forward(pr, PLAIN, **lead), want)
    g3 = backward(pr, PLAIN, want, **lead)
    assert g3[4].shape == lead["gate"].shape and torch.equal(g3[4].reshape(T, K), backward(pr, PLAIN, want)[4])
    for bad in (dict(gate=pr["gate"].reshape(-1)), dict(gate=pr["gate"].reshape(1, -1)), dict(gate=pr["gate"].reshape(-1, 1)),
                dict(idx=pr["idx"].reshape(-1)), dict(x=pr["x"].reshape(2, T // 2, D))):
        with pytest.raises(ValueError):
            forward(pr, PLAIN, **bad)
    for bad in (dict(gate=pr["gate"].reshape(-1)), dict(gate=pr["gate"].reshape(-1, 1)), dict(idx=pr["idx"].reshape(-1))):
        with pytest.raises(ValueError):
            backward(pr, PLAIN, want, **bad)


def test_gate_of_another_type(emu_ops):
    pr = problem(torch.bfloat16)
    want = forward(pr, ADC)
    assert want[2].dtype == torch.bfloat16
    for dt in (torch.float32, torch.float64):
        assert same(forward(pr, ADC, gate=pr["gate"].to(dt)), want)
    assert same(backward(pr, ADC, want, gate=pr["gate"].float()), backward(pr, ADC, want))
    # ADC codes are weighted in the gate's own type
    big = dict(T=T, D=256, E=E, F=256, k=K)
    pr = problem(torch.bfloat16, **big)
    want = forward(pr, ADC)
    got = forward(pr, ADC, gate=pr["gate"].float())
    assert want[2].dtype == torch.uint8 and got[0].dtype == torch.float32 and same(got[1:], want[1:])
    assert torch.equal(got[0].bfloat16(), want[0])
    with pytest.raises(TypeError):
        forward(pr, ADC, gate=pr["gate"].double())


def test_k_tile_bounds_live_until_the_call_returns(emu_ops, monkeypatch):
    """The library reads the bounds through addresses in the packed arguments: a cache that forgets them meanwhile (other
    layers, other threads) must not free them."""
    pr = problem()
    made, alive = [], []
    real, lib = _abi.bounds_array, emu_ops.get_lib()

    def recorded(bounds):
        made.append(weakref.ref(real(bounds)))
        return made[-1]()

    def during(name):
        def call(*args):
            for n in range(1000):
                real((0, n + 1))
            alive.extend(r() is not None for r in made)
            del made[:]
            return getattr(lib, name)(*args)
        return call
    monkeypatch.setattr(_abi, "bounds_array", recorded)
    monkeypatch.setattr(emu_ops, "_LIB", types.SimpleNamespace(
        **{n: during(n) if n in ("amoe_ffn_fwd", "amoe_ffn_bwd", "amoe_router_fwd") else getattr(lib, n) for n in _abi.PROTOTYPES}))
    pr["ir"] = pr["ir"].expand(2, E, 2).contiguous()
    cfg = dataclasses.replace(PLAIN, bounds_up=[0, 16, D])
    backward(pr, cfg, forward(pr, cfg))
    emu_ops.router_fwd(pr["x"], torch.randn(E, D), torch.ones(2), K, [0, 16, D], 1 / 127, -1.0, -1.0)
    assert len(alive) >= 5 and all(alive)


@pytest.mark.parametrize("cfg", [PLAIN, ADC, dataclasses.replace(ADC, noise_std=0.04, noise_per_channel=True)], ids=["plain", "adc", "per_channel"])
def test_weights_in_other_layouts_are_not_copied_where_the_kernels_take_strides(emu_ops, monkeypatch, cfg):
    pr = problem()
    want = forward(pr, cfg)
    turned = {n: pr[n].transpose(1, 2).contiguous().transpose(1, 2) for n in ("keys", "values")}
    wide = {n: torch.cat((pr[n], pr[n]), 2)[:, :, :pr[n].shape[2]] for n in ("keys", "values")}
    packed = []
    real = ffn._abi.FFN_ARGS
    monkeypatch.setattr(ffn._abi, "FFN_ARGS", types.SimpleNamespace(pack=lambda *a: packed.append(a) or real.pack(*a)))
    for layout in (turned, wide):
        got = forward(pr, cfg, **layout)
        for a, b in zip(got, want):
            torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)
        assert layout["keys"].data_ptr() in packed[-1] and layout["values"].data_ptr() in packed[-1]
        back, ref = backward(pr, cfg, got, **layout), backward(pr, cfg, want)
        for a, b in zip(back, ref):
            assert a.is_contiguous()
            torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4)
    assert wide["keys"].data_ptr() in packed[-2]                      # (the backward call before the reference's)
    scattered = pr["keys"].permute(2, 1, 0).contiguous().permute(2, 1, 0)        # neither features nor outputs adjacent
    assert same(forward(pr, cfg, keys=scattered), want)
