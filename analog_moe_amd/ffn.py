"""Fused expert feed-forward of the analog SigmaMoE layer as ONE autograd function.

Same arithmetic as two CVMM calls with a ReLU between them (moe_layer_aihwkit_lightning.py:
384-410, 494-506; cvmm.py:699-897), with the glue folded into the kernels: the ReLU into the
up-projection's store and the down-projection's input gradient, the gate (x) dy outer product
into the weight-gradient loader, the per-position input-range gather into a per-expert table,
and the noise draw into the epilogue.
"""
from __future__ import annotations

import ctypes
from dataclasses import dataclass
from typing import Callable, Optional, Sequence

import torch

from . import _abi, ops, raw


@dataclass
class FFNConfig:
    inp_res: float = -1.0                         # kernel step (1/127 for 8 bit); <= 0 off
    bounds_up: Optional[Sequence[int]] = None     # K-tile bounds of the up-projection
    bounds_down: Optional[Sequence[int]] = None
    out_bound: float = -1.0
    out_res: float = -1.0
    noise_std: float = 0.0                        # in-kernel noise, in units of max|W|
    noise_seed: int = 0
    noise_seed_dev: Optional[torch.Tensor] = None  # int64 device word added to the seed by the kernels
    noise_per_channel: bool = False
    gradient_relative: bool = True
    gradient_scale: float = 1.0
    decay: float = 0.0
    input_min_percentage: float = 0.95
    noise_up: Optional[torch.Tensor] = None       # injected noise [n_tiles, T*k, F] (parity runs)
    noise_down: Optional[torch.Tensor] = None
    wmax_up: Optional[torch.Tensor] = None        # max |W| behind noise and ADC when the weights passed in are
    wmax_down: Optional[torch.Tensor] = None      # modified copies (fp32 [E, 1] or [E, N]); None: taken from them
    seed_bump: int = 0                            # added to noise_seed_dev by the forward's last launch (eager calls
                                                  # only: not among the fields the opaque operators take)
    down_ready: Optional["torch.cuda.Event"] = None  # the down-projection's weights and wmax_down are made on another
                                                  # stream: the current one waits for this event before it reads them
                                                  # (eager calls only, as seed_bump)
    stage_events: Optional[Callable[[bool], int]] = None  # profiling: address of the hipEvent_t pairs recorded around the
                                                  # stages of a direction (argument: backward); eager calls only


CFG_FIELDS = ("inp_res", "bounds_up", "bounds_down", "out_bound", "out_res", "noise_std", "noise_seed",
              "noise_seed_dev", "noise_per_channel", "gradient_relative", "gradient_scale", "decay",
              "input_min_percentage", "noise_up", "noise_down", "wmax_up", "wmax_down")


def cfg_astuple(cfg: FFNConfig) -> tuple:
    """The configuration as positional values, in the order the ``amoe::ffn_fwd`` operator takes them."""
    return tuple(getattr(cfg, f) for f in CFG_FIELDS)


def _n_tiles(bounds) -> int:
    return 1 if bounds is None else len(bounds) - 1


def ir_tables(input_range: Optional[torch.Tensor], E: int, cfg: FFNConfig):
    """Per-expert input ranges of the two projections, fp32: [E, n_tiles_up], [E, n_tiles_down]."""
    if input_range is None:
        return None, None
    ir3 = input_range.detach().float().reshape(2, E, -1)
    return ir3[0, :, :_n_tiles(cfg.bounds_up)].contiguous(), ir3[1, :, :_n_tiles(cfg.bounds_down)].contiguous()


def _p(t: Optional[torch.Tensor]) -> int:
    return 0 if t is None else t.data_ptr()


# What arrives as the kernels want it, which is nearly always, is passed on as it is: a view costs a microsecond of the host.
def _dense(t: torch.Tensor) -> torch.Tensor:
    return t if t.is_contiguous() else t.detach().contiguous()


def _fp32(t: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    return t if t is None or (t.dtype == torch.float32 and t.is_contiguous()) else ops._f32c(t)


def _rows(t: torch.Tensor) -> torch.Tensor:
    """A matrix whose rows are adjacent elements."""
    return t if t.stride(1) == 1 else t.detach().contiguous()


def _operand(w: torch.Tensor) -> torch.Tensor:
    """Weights of a forward product: the kernels take any strides as long as one of the two dimensions is adjacent."""
    _, inner, last = w.stride()
    return w if last == 1 or inner == 1 else w.detach().contiguous()


def _bounds(bounds, K: int):
    """The bounds of a projection's K-tiles as a C array, to be held until the call that reads them returns."""
    b = (0, K) if bounds is None else tuple(map(int, bounds))
    if not 2 <= len(b) <= _abi.AMOE_MAX_TILES + 1:
        raise ValueError(f"number of K-tiles must be in [1, {_abi.AMOE_MAX_TILES}]")
    return _abi.bounds_array(b)


def _pack(cfg: FFNConfig, backward: bool, x, keys, values, input_range, ir_dtype, sel, gate, y, p1, z, z_scale, perm, in_index, offsets, ir_up, ir_dn,
          grads=(0, 0, 0, 0, 0, 0), noise=(None, None), wmax=(None, None), per_channel=False):
    """The argument structure of ``amoe_ffn_fwd`` / ``amoe_ffn_bwd``, and what it points at beside the tensors (to be held
    until the call returns).  All tensors rows-contiguous, x [T, D]."""
    E, D, F = keys.shape
    V = values.shape[2]
    if keys.dtype != x.dtype or values.dtype != x.dtype or gate.dtype != x.dtype:
        raise TypeError("x, keys, values and gate must share one dtype")
    if x.shape[1] != D or values.shape[0] != E or values.shape[1] != F:
        raise ValueError("x / keys / values shapes do not match")
    if x.dtype != torch.float32 and cfg.inp_res > 0:
        raw.check_codes_fit(x.dtype, cfg.inp_res)
    up, down = _bounds(cfg.bounds_up, D), _bounds(cfg.bounds_down, F)
    packed = _abi.FFN_ARGS.pack(
        raw.dtype_code(x), x.shape[0], D, E, F, V, gate.shape[-1],
        x.data_ptr(), x.stride(0), keys.data_ptr(), *keys.stride(), values.data_ptr(), *values.stride(),
        _p(input_range), 0 if ir_dtype is None else raw.code_of(ir_dtype), 0 if input_range is None else input_range.shape[2], sel.data_ptr(), sel.dtype == torch.int64, gate.data_ptr(),
        cfg.inp_res, cfg.out_bound, cfg.out_res, cfg.noise_std,
        len(up) - 1, ctypes.addressof(up), len(down) - 1, ctypes.addressof(down), cfg.noise_seed & 0xFFFFFFFFFFFFFFFF, _p(cfg.noise_seed_dev),
        per_channel, *map(_p, noise), *map(_p, wmax),
        cfg.seed_bump if cfg.noise_seed_dev is not None else 0, 0 if cfg.down_ready is None else cfg.down_ready.cuda_event,
        _p(y), p1.data_ptr(), z.data_ptr(), z.dtype == torch.uint8, _p(z_scale), perm.data_ptr(), in_index.data_ptr(),
        offsets.data_ptr(), _p(ir_up), _p(ir_dn),
        *grads, cfg.gradient_relative, cfg.gradient_scale, cfg.decay, cfg.input_min_percentage,
        0 if cfg.stage_events is None else cfg.stage_events(backward))
    return packed, (up, down)


def _rows_of(t: torch.Tensor, rows: int, cols: int, name: str) -> torch.Tensor:
    """t as a contiguous [rows, cols]."""
    if t.shape == (rows, cols) and t.is_contiguous():
        return t
    if t.dim() == 0 or t.shape[-1] != cols or t.numel() != rows * cols:
        raise ValueError(f"{name} must be [{rows}, {cols}], not {tuple(t.shape)}")
    return t.detach().reshape(rows, cols).contiguous()


def _check_heads(sel: torch.Tensor, gate: torch.Tensor, M: int, k: int) -> None:
    """The library counts the heads once for both."""
    if sel.numel() != M or gate.numel() != M or sel.shape[-1] != k or gate.shape[-1] != k:
        raise ValueError(f"sel_idx and gate must hold k values per token: {tuple(sel.shape)} and {tuple(gate.shape)}")


def _int_ids(sel_idx: torch.Tensor) -> torch.Tensor:
    if sel_idx.dtype not in (torch.int32, torch.int64):
        sel_idx = sel_idx.detach().to(torch.int64)
    return _dense(sel_idx)


def _range_table(input_range: torch.Tensor, E: int, cfg: FFNConfig) -> torch.Tensor:
    """The parameter as the library reads it, [2, E, columns].  Types it does not know are converted, but for the launch that makes the
    range tables together with max |W| and takes the parameter as it is (TypeError)."""
    shape = input_range.shape
    if len(shape) != 3 or shape[0] != 2 or shape[1] != E:
        input_range = input_range.detach().reshape(2, E, -1)
    if input_range.dtype in raw.DTYPE_CODES or (_reads_wmax(cfg) and cfg.wmax_up is None and not cfg.noise_per_channel):
        raw.dtype_code(input_range)
        return _dense(input_range)
    return _dense(input_range.detach().float())


def _noise(t: Optional[torch.Tensor], bounds, M: int, N: int) -> Optional[torch.Tensor]:
    """Injected output noise of a projection, fp32 [K-tiles, M, N]."""
    if t is None:
        return None
    if t.numel() != _n_tiles(bounds) * M * N:
        raise ValueError(f"injected noise must be [{_n_tiles(bounds)}, {M}, {N}], not {tuple(t.shape)}")
    return _fp32(t)


def _reads_wmax(cfg: FFNConfig) -> bool:
    return cfg.out_bound > 0 or (cfg.noise_std > 0 and cfg.noise_up is None)


def _wmax_tables(cfg: FFNConfig, keys: torch.Tensor, values: torch.Tensor):
    """The caller's max |W| tables as the library takes them (fp32; None: it makes them) and whether they have a column per
    output channel.  Each table says for itself whether it is [E] or [E, N]; the library has one flag for both."""
    if not _reads_wmax(cfg):
        return (None, None), False
    if cfg.wmax_up is None:
        if keys.is_contiguous() and values.is_contiguous():
            return (None, None), cfg.noise_per_channel
        # (the library's own reduction walks dense weights)
        return tuple(ops.weight_abs_max(w, cfg.noise_per_channel) for w in (keys, values)), cfg.noise_per_channel
    E = keys.shape[0]
    given = ((cfg.wmax_up, keys.shape[2]), (cfg.wmax_down, values.shape[2]))
    if any(t is None or t.numel() // E not in (1, N) for t, N in given):
        raise ValueError("max |W| tables must be [E] or [E, output channels]")
    wide = [t.numel() // E == N != 1 for t, N in given]
    late = cfg.wmax_down
    if cfg.down_ready is not None and (late.dtype != torch.float32 or not late.is_contiguous() or wide[0] != wide[1]):
        torch.cuda.current_stream().wait_event(cfg.down_ready)
    tables = [_fp32(t) for t, _ in given]
    if any(wide):
        tables = [t if w else t.reshape(-1)[:E, None].expand(E, N).contiguous() for t, w, (_, N) in zip(tables, wide, given)]
    return tuple(tables), any(wide)


def ffn_forward(x, keys, values, input_range, gate, sel_idx, cfg: FFNConfig):
    """Sort, both projections and the gate reduction (``amoe_ffn_fwd``).  Returns (y, p1, z, perm, in_index, offsets,
    z_scale, ir_up, ir_dn): the result and what the backward pass reads again.  z is the down-projection's k-head result
    [T*k, D], either as values (z_scale empty) or as uint8 ADC codes with z_scale [E, 2] (``ops.dequant_codes``)."""
    ops._need_gpu(x, keys, values, input_range, gate, sel_idx, cfg.noise_up, cfg.noise_down, cfg.wmax_up, cfg.wmax_down,
                  cfg.noise_seed_dev)
    if x.dim() != 2:
        raise ValueError("x must be [tokens, features]")
    lib = ops.get_lib()
    if cfg.down_ready is not None and not values.is_contiguous():    # (torch may read them below)
        torch.cuda.current_stream().wait_event(cfg.down_ready)
    x, keys, values, own_gate = _rows(x), _operand(keys), _operand(values), _dense(gate)
    gate = own_gate if own_gate.dtype == x.dtype else own_gate.detach().to(x.dtype)
    sel = _int_ids(sel_idx)
    dev, dt = x.device, x.dtype
    (E, D, F), V = keys.shape, values.shape[2]
    T, k = x.shape[0], sel.shape[-1]
    M = T * k
    _check_heads(sel, gate, M, k)
    if cfg.noise_seed_dev is not None and (cfg.noise_seed_dev.dtype != torch.int64 or cfg.noise_seed_dev.numel() != 1):
        raise ValueError("noise_seed_dev must be one int64 word")
    noise = _noise(cfg.noise_up, cfg.bounds_up, M, F), _noise(cfg.noise_down, cfg.bounds_down, M, V)
    wmax, per_channel = _wmax_tables(cfg, keys, values)
    y, p1 = x.new_empty((T, V)), x.new_empty((M, F))
    perm, in_index = (torch.empty(M, dtype=torch.int32, device=dev) for _ in range(2))
    offsets = torch.empty(E + 1, dtype=torch.int32, device=dev)
    ir_up = ir_dn = None
    if input_range is not None:
        input_range = _range_table(input_range, E, cfg)
        ir_up, ir_dn = (torch.empty((E, _n_tiles(b)), dtype=torch.float32, device=dev)
                        for b in (cfg.bounds_up, cfg.bounds_down))
    chain = input_range is not None and cfg.inp_res > 0 and _n_tiles(cfg.bounds_down) == 1
    codes = chain and z_as_codes(p1, values, cfg)
    if codes and gate is not own_gate:               # (codes are weighted in the gate's type)
        raw.dtype_code(own_gate)
    z = torch.empty((M, V), dtype=torch.uint8 if codes else dt, device=dev)
    z_scale = torch.empty((E, 2) if codes else 0, dtype=torch.float32, device=dev)
    if M == 0:                                       # no tokens: nothing to launch but the step counter
        if cfg.seed_bump and cfg.noise_seed_dev is not None:
            cfg.noise_seed_dev.add_(cfg.seed_bump)
        if input_range is not None:
            ir_up, ir_dn = ir_tables(input_range, E, cfg)
        return y, p1, z, perm, in_index, offsets.zero_(), z_scale, ir_up, ir_dn
    args, held = _pack(cfg, False, x, keys, values, input_range, None if input_range is None else input_range.dtype, sel, gate,
                 y, p1, z, z_scale, perm, in_index, offsets, ir_up, ir_dn, noise=noise, wmax=wmax,
                 per_channel=per_channel)
    ws = torch.empty(lib.amoe_ffn_fwd_workspace(args), dtype=torch.uint8, device=dev)
    _abi.check(lib, lib.amoe_ffn_fwd(args, ws.data_ptr(), ws.numel(), ops._stream(x), None), "amoe_ffn_fwd")
    del held
    if codes and gate is not own_gate:
        y = ops.gate_reduce_codes(z, z_scale, sel, own_gate)
    return y, p1, z, perm, in_index, offsets, z_scale, ir_up, ir_dn


def z_as_codes(p1q: torch.Tensor, values: torch.Tensor, cfg: FFNConfig) -> bool:
    """Whether the down-projection leaves its result as ADC codes (a pure function of shapes and settings)."""
    return ops.codes_supported(p1q, values, ir_by_expert=True, inp_res=cfg.inp_res, n_tiles=_n_tiles(cfg.bounds_down),
                               out_bound=cfg.out_bound, out_res=cfg.out_res, noise=cfg.noise_down,
                               per_channel=cfg.noise_per_channel)


def ffn_backward(dy, x, keys, values, gate, sel_idx, p1, z, z_scale, perm, in_index, offsets, ir_up, ir_dn,
                 cfg: FFNConfig, want_ir_grad: bool, ir_dtype: torch.dtype = torch.float32):
    """Returns (grad_x, grad_keys, grad_values, grad_ir [2, E, n_tiles] of type ir_dtype or None, grad_gate)
    (``amoe_ffn_bwd``)."""
    ops._need_gpu(dy, x, keys, values, gate, sel_idx, p1, z, z_scale, perm, in_index, offsets, ir_up, ir_dn)
    lib = ops.get_lib()
    if x.dim() != 2:
        x = x.detach().reshape(-1, x.shape[-1])
    x = _rows(x)
    keys, values = (w if w.stride(2) == 1 else w.detach().contiguous() for w in (keys, values))
    gate_c, sel = _dense(gate), _int_ids(sel_idx)
    if gate_c.dtype != x.dtype:
        gate_c = gate_c.detach().to(x.dtype)
    (E, D, F), V = keys.shape, values.shape[2]
    T, k = x.shape[0], gate.shape[-1]
    M = T * k
    _check_heads(sel, gate, M, k)
    # what the forward call left may come back through hooks in another layout, and from a caller as anything
    dy, p1, z = _rows_of(dy, T, V, "dy"), _rows_of(p1, M, F, "p1"), _rows_of(z, M, V, "z")
    if dy.dtype != x.dtype or p1.dtype != x.dtype or z.dtype not in (x.dtype, torch.uint8):
        raise TypeError("dy, p1 and x must share one dtype, z that or uint8 codes")
    if z.dtype == torch.uint8 and (z_scale.dtype != torch.float32 or tuple(z_scale.shape) != (E, 2) or not z_scale.is_contiguous()):
        raise ValueError("ADC codes come with their scale, fp32 [E, 2]")
    for t, n, name in ((perm, M, "perm"), (in_index, M, "in_index"), (offsets, E + 1, "offsets")):
        if raw._i32(t, name).numel() != n:
            raise ValueError(f"{name} must hold {n} values")
    if (ir_up is None) != (ir_dn is None):
        raise ValueError("input ranges of both projections or of none")
    ir_up, ir_dn = _fp32(ir_up), _fp32(ir_dn)
    if ir_up is not None and (ir_up.shape != (E, _n_tiles(cfg.bounds_up)) or ir_dn.shape != (E, _n_tiles(cfg.bounds_down))):
        raise ValueError("input ranges must be [E, K-tiles of the projection]")
    grad_x = x.new_empty(x.shape)
    grad_keys, grad_values, grad_gate = keys.new_empty((E, D, F)), values.new_empty((E, F, V)), torch.empty_like(gate_c)
    grad_ir = None
    if ir_up is not None and want_ir_grad:
        grad_ir = torch.empty((2, E, max(ir_up.shape[1], ir_dn.shape[1])), dtype=ir_dtype, device=x.device)
    if perm.numel() == 0:
        for g in (grad_x, grad_keys, grad_values, grad_gate, grad_ir):
            if g is not None:
                g.zero_()
        return grad_x, grad_keys, grad_values, grad_ir, grad_gate
    args, held = _pack(cfg, True, x, keys, values, None, None if grad_ir is None else ir_dtype, sel, gate_c, None, p1, z, z_scale, perm, in_index, offsets,
                 ir_up, ir_dn, (dy.data_ptr(), grad_x.data_ptr(), grad_keys.data_ptr(), grad_values.data_ptr(),
                                grad_gate.data_ptr(), _p(grad_ir)))
    ws = torch.empty(lib.amoe_ffn_bwd_workspace(args), dtype=torch.uint8, device=x.device)
    _abi.check(lib, lib.amoe_ffn_bwd(args, ws.data_ptr(), ws.numel(), ops._stream(x), ops._side(x)), "amoe_ffn_bwd")
    del held
    return grad_x, grad_keys, grad_values, grad_ir, grad_gate


class AnalogMoEFFN(torch.autograd.Function):
    """y[t] = sum_j gate[t,j] * A(relu(A(x[t], keys[e_tj])), values[e_tj]).
    input_range: [2, E, n_tiles] (row 0 up-, row 1 down-projection) or None."""

    @staticmethod
    def forward(ctx, x, keys, values, input_range, gate, sel_idx, cfg: FFNConfig):
        y, p1, z, perm, in_index, offsets, z_scale, ir_up, ir_dn = ffn_forward(x, keys, values, input_range, gate,
                                                                               sel_idx, cfg)
        ctx.save_for_backward(x, keys, values, gate, sel_idx, p1, z, z_scale, perm, in_index, offsets, ir_up, ir_dn)
        ctx.cfg = cfg
        ctx.ir_shape = None if input_range is None else input_range.shape
        ctx.ir_dtype = None if input_range is None else input_range.dtype
        return y

    @staticmethod
    def backward(ctx, dy):
        x, keys, values, gate, sel_idx, p1, z, z_scale, perm, in_index, offsets, ir_up, ir_dn = ctx.saved_tensors
        grad_x, grad_keys, grad_values, grad_ir, grad_gate = ffn_backward(
            dy, x, keys, values, gate, sel_idx, p1, z, z_scale, perm, in_index, offsets, ir_up, ir_dn, ctx.cfg,
            ctx.needs_input_grad[3], ctx.ir_dtype or torch.float32)
        if grad_ir is not None:
            grad_ir = grad_ir.reshape(ctx.ir_shape)
        return grad_x, grad_keys, grad_values, grad_ir, grad_gate, None, None


def moe_ffn(x, keys, values, input_range, gate, sel_idx, cfg: FFNConfig) -> torch.Tensor:
    """The fused expert feed-forward.  Eagerly this is ``AnalogMoEFFN``; while ``torch.compile`` traces,
    the same two functions are reached through the opaque operators ``amoe::ffn_fwd`` / ``amoe::ffn_bwd``
    (their side streams and ctypes calls are nothing a tracer can follow)."""
    if torch.compiler.is_compiling():
        return torch.ops.amoe.ffn_fwd(x, keys, values, input_range, gate, sel_idx, *cfg_astuple(cfg))[0]
    if not torch.is_grad_enabled() and ops.unwatched():
        return ffn_forward(x, keys, values, input_range, gate, sel_idx, cfg)[0]
    return AnalogMoEFFN.apply(x, keys, values, input_range, gate, sel_idx, cfg)
