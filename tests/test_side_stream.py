"""The layer calls' second stream is joined however a call ends: what its launches read and write belongs to the caller again
once the call has returned, with an error as without one."""
import ctypes

import torch

from analog_moe_amd import ffn
from tests.test_emu_kernels import emu_ops  # noqa: F401

MAIN, SIDE = 11, 12                      # stream handles: the host build only writes down what is given to them


def arguments(T, D, E, F, k, cfg, grads=(0, 0, 0, 0, 0, 0)):
    g = torch.Generator().manual_seed(1)
    M = T * k
    t = dict(x=torch.randn(T, D, generator=g), keys=torch.randn(E, D, F, generator=g), values=torch.randn(E, F, D, generator=g),
             gate=torch.rand(T, k, generator=g), sel=torch.randint(0, E, (M + 1,), generator=g, dtype=torch.int64), y=torch.zeros(T, D),
             p1=torch.rand(M, F, generator=g), z=torch.rand(M, D, generator=g), perm=torch.arange(M, dtype=torch.int32),
             in_index=(torch.arange(M) // k).int(), offsets=(torch.arange(E + 1) * M // E).int())
    args, t["held"] = ffn._pack(cfg, any(grads), t["x"], t["keys"], t["values"], None, None, t["sel"], t["gate"], t["y"], t["p1"], t["z"], None,
                     t["perm"], t["in_index"], t["offsets"], None, None, grads)
    return t, args


def streams(lib):
    count = {}
    for name, n in (("amoe_emu_launches", 1), ("amoe_emu_not_waited_for", 2)):
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = ctypes.c_longlong, [ctypes.c_void_p] * n
        count[name] = fn
    return count["amoe_emu_launches"], count["amoe_emu_not_waited_for"]


def shifted(args, ptr, by):
    """The packed arguments with a pointer moved."""
    at = args.index(ptr.to_bytes(8, "little"))
    return args[:at] + (ptr + by).to_bytes(8, "little") + args[at + 8:]


def test_forward(emu_ops):
    """nothing beside the first stream, however large the weights"""
    lib = emu_ops.get_lib()
    launches, not_waited = streams(lib)
    t, args = arguments(1, 6144, 1, 512, 1, ffn.FFNConfig(inp_res=-1.0, out_bound=12.0, out_res=254.0))
    assert t["keys"].nbytes + t["values"].nbytes >= 24 << 20
    ws = torch.empty(lib.amoe_ffn_fwd_workspace(args), dtype=torch.uint8)
    before = launches(SIDE)
    rc = lib.amoe_ffn_fwd(args, ws.data_ptr(), ws.numel(), MAIN, SIDE)
    assert rc == 0 and launches(SIDE) == before and not_waited(MAIN, SIDE) == 0


def backward_arguments(T=260, D=6144, E=1, F=4, k=2):
    """A call whose k-head tensors are large enough for the second stream, and its weight gradient of the values."""
    out = [torch.zeros(n) for n in (T * D, E * D * F, E * F * D + 1, T * k)]
    dy = torch.randn(T, D)
    ptrs = [t.data_ptr() for t in (dy, *out)] + [0]
    t, args = arguments(T, D, E, F, k, ffn.FFNConfig(inp_res=-1.0), ptrs)
    return (t, out, dy), args, out[2]


def test_backward(emu_ops):
    """the streaming companions beside the weight gradients, which refuse an output that is not aligned to its elements"""
    lib = emu_ops.get_lib()
    launches, not_waited = streams(lib)
    held, args, grad_values = backward_arguments()
    args = shifted(args, grad_values.data_ptr(), 2)
    ws = torch.empty(lib.amoe_ffn_bwd_workspace(args), dtype=torch.uint8)
    before = launches(SIDE)
    rc = lib.amoe_ffn_bwd(args, ws.data_ptr(), ws.numel(), MAIN, SIDE)
    assert rc != 0 and launches(SIDE) == before + 2 and not_waited(MAIN, SIDE) == 0


def test_events_that_cannot_be_made(emu_ops):
    """without both of its events the second stream is given nothing, as nothing could be made to wait for it later"""
    lib = emu_ops.get_lib()
    launches, not_waited = streams(lib)
    lib.amoe_emu_allow_events.argtypes, lib.amoe_emu_allow_events.restype = [ctypes.c_longlong], None
    held, args, _ = backward_arguments()
    ws = torch.empty(lib.amoe_ffn_bwd_workspace(args), dtype=torch.uint8)
    before = launches(SIDE)
    lib.amoe_emu_allow_events(1)
    try:
        rc = lib.amoe_ffn_bwd(args, ws.data_ptr(), ws.numel(), MAIN, SIDE)
    finally:
        lib.amoe_emu_allow_events(-1)
    assert rc > 0 and launches(SIDE) == before and not_waited(MAIN, SIDE) == 0
