"""The operations the parts are written against, bound to the gfx950 kernel library.

Every function checks shapes, dtypes, contiguity and device on the host before a
kernel is launched (a kernel never sees an operand it was not written for), then
calls the library's C entry point on the current stream.  There is no CPU path:
without the compiled library or without a GPU the first call raises.

Tests may install another backend with ``set_backend`` (an object with the same
functions) to exercise the engine's bookkeeping on the host; nothing in the
product does.
"""
from __future__ import annotations

import ctypes
import os
import re
from typing import Optional

import torch

_F32, _BF16 = 0, 1
_backend = None


def set_backend(backend) -> None:
    """Install an object providing this module's functions (tests only); None restores the library."""
    global _backend
    _backend = backend


class KernelError(RuntimeError):
    pass


_C_TYPES = {"int": ctypes.c_int, "unsigned": ctypes.c_uint, "size_t": ctypes.c_size_t, "float": ctypes.c_float, "double": ctypes.c_double,
            "long": ctypes.c_long, "long long": ctypes.c_longlong, "unsigned long long": ctypes.c_ulonglong}


def entry_points() -> dict:
    """name -> (result type, argument types) of the library's C entry points, from the declarations in the sources that it is built from."""
    from ..csrc.build import sources
    out = {}
    for path in sources():
        with open(path, encoding="utf-8") as f:
            text = re.sub(r"//[^\n]*", "", f.read())
        for result, name, args in re.findall(r'extern "C"\s+([\w\s]+?[\s\*]+)(tp_\w+)\s*\(([^)]*)\)\s*\{', text):
            result = " ".join(result.split())
            types = []
            for arg in args.split(",") if args.strip() not in ("", "void") else ():
                kind = "*" if "*" in arg or "hipStream_t" in arg else " ".join(w for w in arg.split()[:-1] if w != "const")
                types.append(ctypes.c_void_p if kind == "*" else _C_TYPES[kind])
            out[name] = (ctypes.c_char_p if "*" in result else None if result == "void" else _C_TYPES[result], types)
    return out


def _declare(lib) -> None:
    # (addresses, numbers and None go to a declared entry point as they are; undeclared ones want an object of ctypes for each, which costs a
    # launch of a dozen tensors more than the launch itself)
    for name, (result, args) in entry_points().items():
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = result, args


class _Library:
    """The compiled kernel library, loaded on first use."""

    _lib = None

    @classmethod
    def get(cls):
        if cls._lib is None:
            if not torch.cuda.is_available():
                raise KernelError("tempura_amd needs a GPU: torch.cuda.is_available() is False and there is no CPU path")
            from ..csrc.build import ensure_built
            path = ensure_built()
            try:
                lib = ctypes.CDLL(path)
            except OSError as e:
                raise KernelError(f"cannot load the kernel library {path}: {e}") from e
            _declare(lib)
            cls._lib = lib
            cls.path = path
        return cls._lib


def library():
    return _Library.get()


class KernelTimer:
    """Times every call into the kernel library made while it is active (``with KernelTimer() as t:``), with a pair
    of events on the current stream around each call: eager steps only (events cannot be recorded into a graph
    that is replayed), and the pairs serialise nothing, so a call's time includes what its kernels wait for.
    ``label`` (settable at any time) is stored with every call; ``table()`` waits for the device and returns
    rows (entry point, label, calls, total microseconds), largest first."""

    def __init__(self):
        self.label = ""
        self._events = []

    def __enter__(self):
        global _timer
        self._before, _timer = _timer, self
        return self

    def __exit__(self, *exc):
        global _timer
        _timer = self._before
        return False

    def table(self, by_label: bool = False):
        torch.cuda.synchronize()
        total = {}
        for name, label, e0, e1 in self._events:
            key = (name, label if by_label else "")
            calls, us = total.get(key, (0, 0.0))
            total[key] = (calls + 1, us + 1e3 * e0.elapsed_time(e1))
        return sorted(((k[0], k[1], c, us) for k, (c, us) in total.items()), key=lambda r: -r[3])


_timer: Optional[KernelTimer] = None


def _call(name: str, *args, tag: Optional[tuple] = None) -> None:
    """``tag``: what distinguishes this call in a ``KernelTimer``'s table (a product's sizes)."""
    lib = _Library.get()
    t = _timer
    if t is not None:
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
    rc = getattr(lib, name)(*args)
    if rc != 0:
        raise KernelError(f"{name}: {lib.tp_last_error().decode()}")
    if t is not None:
        e1.record()
        t._events.append((name if tag is None else name + " " + "x".join(map(str, tag)), t.label, e0, e1))


def _dt(t: torch.Tensor) -> int:
    if t.dtype == torch.float32:
        return _F32
    if t.dtype == torch.bfloat16:
        return _BF16
    raise KernelError(f"unsupported dtype {t.dtype}")


def _dtcode(dtype: torch.dtype) -> int:
    if dtype == torch.float32:
        return _F32
    if dtype == torch.bfloat16:
        return _BF16
    raise KernelError(f"unsupported dtype {dtype}")


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_raw_device = getattr(torch._C, "_cuda_getDevice", None) or torch.cuda.current_device


def _stream():
    """The current stream's handle (of the current device).  Asked for at every launch: the direct call is
    some 8 us cheaper than ``torch.cuda.current_stream()``, a quarter of an eager launch's host time."""
    if _raw_stream is not None:
        return _raw_stream(_raw_device())
    return torch.cuda.current_stream().cuda_stream


def _need(cond: bool, msg: str) -> None:
    if not cond:
        raise KernelError(msg)


def _dev_ok(*ts) -> None:
    for t in ts:
        if t is not None:
            if not t.is_cuda:
                raise KernelError("operand is not on the GPU")
            if not t.is_contiguous():
                raise KernelError("operand is not contiguous")


def _i32(t: torch.Tensor, n: int, what: str) -> None:
    if not (t.dtype == torch.int32 and t.numel() >= n and t.dim() >= 1):
        raise KernelError(f"{what}: need int32 with {n} elements")


# ---------------------------------------------------------------------------------
def embed(tokens: torch.Tensor, table: torch.Tensor, positions: Optional[torch.Tensor] = None,
          inv_freq: Optional[torch.Tensor] = None, streams: int = 1) -> torch.Tensor:
    """int32 [n] , [vocab, hidden] -> float32 [n, hidden]; with ``streams`` > 1, [n, streams * hidden] holding that
    many copies of each row.  With ``inv_freq`` (float64 [ceil(hidden / 2)]) and ``positions`` (int32 [n]) a
    sinusoidal position vector is added: element 2i gets sin(p * inv_freq[i]), element 2i + 1 the cosine."""
    if _backend is not None:
        if inv_freq is None and streams == 1:
            return _backend.embed(tokens, table)
        return _backend.embed(tokens, table, positions, inv_freq, streams)
    _dev_ok(tokens, table, positions, inv_freq)
    n = tokens.numel()
    _i32(tokens, n, "embed tokens")
    _need(table.dim() == 2, "embed: table must be [vocab, hidden]")
    hidden = table.shape[1]
    if inv_freq is None and streams == 1:
        out = torch.empty((n, hidden), dtype=torch.float32, device=table.device)
        _call("tp_embed", _ptr(tokens), _ptr(table), _dt(table), _ptr(out), n, hidden, _stream())
        return out
    _need(streams >= 1, "embed: streams must be positive")
    if inv_freq is not None:
        _need(positions is not None, "embed: positions missing")
        _i32(positions, n, "embed positions") if n else None
        _need(inv_freq.dtype == torch.float64 and inv_freq.numel() == (hidden + 1) // 2, "embed: inv_freq must be float64 [ceil(hidden / 2)]")
    out = torch.empty((n, streams * hidden), dtype=torch.float32, device=table.device)
    _call("tp_embed_pos", _ptr(tokens), _ptr(positions), _ptr(table), _dt(table), _ptr(inv_freq), _ptr(out), n, hidden,
          int(streams), _stream())
    return out


def stream_step(h: torch.Tensor, streams: int, y: Optional[torch.Tensor] = None, mix: Optional[torch.Tensor] = None,
                out_coef: Optional[torch.Tensor] = None, in_coef: Optional[torch.Tensor] = None,
                norm_weight: Optional[torch.Tensor] = None, eps: float = 0.0, out_dtype: Optional[torch.dtype] = None,
                rows: Optional[torch.Tensor] = None, write_back: bool = True) -> Optional[torch.Tensor]:
    """One step of ``streams`` copies of the residual stream, h float32 [n, streams * width], per row:
    with ``y`` (float32 [n, width], a sublayer's output) every stream b becomes sum_a mix[a, b] h[a] + out_coef[b] * y
    (``mix`` float32 [streams, streams], None: identity; ``out_coef`` [streams], None: ones), written back into
    ``h`` when ``write_back``; then, with ``out_dtype``, the result is u = sum_a in_coef[a] h[a] (None: the plain
    sum), normed with ``norm_weight`` (float32 [width]; u / sqrt(mean(u^2) + eps) * weight) when that is given,
    as ``out_dtype`` [n or len(rows), width].  ``rows`` (int32) picks the rows."""
    if _backend is not None:
        return _backend.stream_step(h, streams, y, mix, out_coef, in_coef, norm_weight, eps, out_dtype, rows, write_back)
    _dev_ok(h, y, mix, out_coef, in_coef, norm_weight, rows)
    _need(h.dtype == torch.float32 and h.dim() == 2 and streams >= 1 and h.shape[1] % streams == 0,
          "stream_step: h must be float32 [n, streams * width]")
    n, width = h.shape[0], h.shape[1] // streams
    if y is not None:
        _need(y.dtype == torch.float32 and tuple(y.shape) == (n, width), "stream_step: y must be float32 [n, width]")
    for t, size, what in ((mix, streams * streams, "mix"), (out_coef, streams, "out_coef"), (in_coef, streams, "in_coef"),
                          (norm_weight, width, "norm_weight")):
        if t is not None:
            if not (t.dtype == torch.float32 and t.numel() == size):
                raise KernelError(f"stream_step: {what} must be float32 with {size} elements")
    n_out = n
    if rows is not None:
        n_out = rows.numel()
        _i32(rows, n_out, "stream_step rows") if n_out else None
        _need(not (write_back and y is not None) or out_dtype is None, "stream_step: a step over chosen rows cannot write all streams back")
    out = None
    if out_dtype is not None:
        out = torch.empty((n_out, width), dtype=out_dtype, device=h.device)
        if n_out == 0:
            return out          # (a step in which no row is wanted)
    else:
        _need(y is not None and write_back, "stream_step: nothing to do")
    _call("tp_hc_step", _ptr(h), _ptr(y), _ptr(mix), _ptr(out_coef), _ptr(in_coef), _ptr(norm_weight), float(eps),
          _ptr(out), _dtcode(out_dtype) if out_dtype is not None else _F32, _ptr(rows), n_out, int(streams), width,
          int(bool(write_back) and y is not None), _stream())
    return out


def scale_(x: torch.Tensor, scale: float) -> torch.Tensor:
    """x *= scale in place (float32)."""
    if _backend is not None:
        return _backend.scale_(x, scale)
    _dev_ok(x)
    _need(x.dtype == torch.float32, "scale_: needs float32")
    _call("tp_scale_f32", _ptr(x), int(x.numel()), float(scale), _stream())
    return x


def gated_act(gu: torch.Tensor, out_dtype: torch.dtype, slope: float = 1.0, limit: float = 0.0, up_offset: float = 0.0,
              interleaved: bool = False) -> torch.Tensor:
    """[m, 2i] (gate columns then up columns; ``interleaved``: eight gate and eight up columns in turn, the layout of
    ``interleave_gate_up``; no part asks for it, it is what the products that gate their own sums are tested against)
    -> out_dtype [m, i]: g = min(gate, limit), u = clamp(up, -limit, limit) (limit <= 0: none),
    g * sigmoid(slope * g) * (u + up_offset)."""
    if _backend is not None:
        return _backend.gated_act(gu, out_dtype, slope, limit, up_offset, interleaved)
    _dev_ok(gu)
    _need(gu.dim() == 2 and gu.shape[1] % 2 == 0, "gated_act: input must be [m, 2i]")
    m, i2 = gu.shape
    out = torch.empty((m, i2 // 2), dtype=out_dtype, device=gu.device)
    _call("tp_gated_act", _ptr(gu), _dt(gu), _ptr(out), _dtcode(out_dtype), m, i2 // 2, float(slope),
          float(limit), float(up_offset), int(bool(interleaved)), _stream())
    return out


def qk_store(rows: torch.Tensor, q_bias: Optional[torch.Tensor], k_bias: Optional[torch.Tensor], slots: Optional[torch.Tensor],
             num_heads: int, num_kv_heads: int, head_dim: int, k_cache: Optional[torch.Tensor],
             v_cache: Optional[torch.Tensor], q_dtype: torch.dtype) -> torch.Tensor:
    """float32 rows [n, (heads + kv_heads) * head_dim] of a projection (no rotation): biases (float32, per column)
    are added, q is returned as q_dtype [n, heads, head_dim], k goes to the cache rows ``slots`` of ``k_cache`` and,
    when ``v_cache`` is given (values that are the keys), into the transposed value cache too.  ``slots`` None: the
    rows hold q only."""
    if _backend is not None:
        return _backend.qk_store(rows, q_bias, k_bias, slots, num_heads, num_kv_heads, head_dim, k_cache, v_cache, q_dtype)
    _dev_ok(rows, q_bias, k_bias, slots, k_cache, v_cache)
    _need(rows.dtype == torch.float32 and rows.dim() == 2, "qk_store: rows must be float32 [n, width]")
    n = rows.shape[0]
    width = (num_heads + (num_kv_heads if slots is not None else 0)) * head_dim
    if not (rows.shape[1] == width):
        raise KernelError(f"qk_store: row width {rows.shape[1]} != {width}")
    for b, size in ((q_bias, num_heads * head_dim), (k_bias, num_kv_heads * head_dim)):
        if b is not None:
            _need(b.dtype == torch.float32 and b.numel() == size, "qk_store: bias must be float32, one value per column")
    page_size, cache_dt = 1, _F32
    if slots is not None:
        _i32(slots, n, "slots") if n else None
        _need(k_cache is not None and k_cache.dim() == 4 and k_cache.shape[1] == num_kv_heads and k_cache.shape[3] == head_dim,
              "qk_store: k cache must be [pages, kv_heads, page_size, head_dim]")
        page_size, cache_dt = k_cache.shape[2], _dt(k_cache)
        if v_cache is not None:
            _need(tuple(v_cache.shape) == (k_cache.shape[0], num_kv_heads, head_dim, page_size) and v_cache.dtype == k_cache.dtype,
                  "qk_store: v cache must be [pages, kv_heads, head_dim, page_size] of the key cache's type")
    q = torch.empty((n, num_heads, head_dim), dtype=q_dtype, device=rows.device)
    _call("tp_qk_store", _ptr(rows), rows.shape[1], _ptr(q_bias), _ptr(k_bias), _ptr(slots), n, num_heads, num_kv_heads, head_dim,
          _ptr(q), _dtcode(q_dtype), _ptr(k_cache if slots is not None else None), _ptr(v_cache if slots is not None else None),
          cache_dt, page_size, _stream())
    return q


def causal_conv(proj: torch.Tensor, col0: int, channels: int, weight: torch.Tensor, bias: Optional[torch.Tensor], state: torch.Tensor,
                cu_seqlens: torch.Tensor, token_req: torch.Tensor, state_slots: torch.Tensor, num_requests: int,
                state_off: int = 0, act: bool = True, max_run: int = 0) -> torch.Tensor:
    """Causal convolution per channel over each request's run of tokens, then SiLU (``act`` False: the sums
    themselves).  ``proj`` float32 [n, width] holds the inputs at columns col0 .. col0 + channels; ``weight``
    [taps, channels] (tap-major; the last tap is the current token's), ``bias`` [channels] or None; ``state`` float32
    [slots, row] whose rows hold, from element ``state_off`` on, the carried inputs [taps - 1, channels] (oldest
    first) of the request in that slot: they are read for the first tokens of a run and replaced by the run's last
    inputs.  ``max_run``: the longest run (0: not known); runs of one token are one launch.  Returns float32 [n, channels]."""
    if _backend is not None:
        if state_off == 0 and act and bias is not None:
            return _backend.causal_conv(proj, col0, channels, weight, bias, state, cu_seqlens, token_req, state_slots, num_requests)
        return _backend.causal_conv(proj, col0, channels, weight, bias, state, cu_seqlens, token_req, state_slots, num_requests,
                                    state_off, act)
    _dev_ok(proj, weight, bias, state, cu_seqlens, token_req, state_slots)
    _need(proj.dtype == torch.float32 and proj.dim() == 2 and 0 <= col0 and col0 + channels <= proj.shape[1], "causal_conv: bad rows")
    _need(weight.dtype == torch.float32 and weight.dim() == 2 and weight.shape[1] == channels, "causal_conv: weight must be float32 [taps, channels]")
    taps = weight.shape[0]
    _need(bias is None or (bias.dtype == torch.float32 and bias.numel() == channels), "causal_conv: bias must be float32 [channels]")
    _need(state.dtype == torch.float32 and state.dim() == 2 and state_off >= 0 and state.shape[1] >= state_off + (taps - 1) * channels,
          "causal_conv: state rows too short")
    n = proj.shape[0]
    _i32(cu_seqlens, num_requests + 1, "cu_seqlens")
    _i32(state_slots, num_requests, "state_slots")
    _i32(token_req, n, "token_req") if n else None
    out = torch.empty((n, channels), dtype=torch.float32, device=proj.device)
    _call("tp_causal_conv", _ptr(proj), proj.shape[1], int(col0), _ptr(weight), _ptr(bias), _ptr(state),
          int(state.shape[1]), int(state_off), _ptr(cu_seqlens), _ptr(token_req), _ptr(state_slots), _ptr(out),
          n, int(num_requests), channels, taps, int(bool(act)), int(max_run), _stream())
    return out


def ssm_scan(xbc: torch.Tensor, proj: torch.Tensor, dt_col0: int, dt_bias: torch.Tensor, a_log: torch.Tensor, d_skip: torch.Tensor,
             state: torch.Tensor, state_off: int, cu_seqlens: torch.Tensor, state_slots: torch.Tensor, num_requests: int,
             num_heads: int, head_dim: int, state_size: int, groups: int, max_run: Optional[int] = None) -> torch.Tensor:
    """The selective recurrence per head over each request's run: with dt = softplus(proj[:, dt_col0 + h] + dt_bias[h])
    and a = exp(-exp(a_log[h]) * dt):  S <- a S + dt B x^T,  y = S^T C + d_skip[h] x.  ``xbc`` float32 [n, channels]
    holds x [heads * head_dim] | B [groups * state] | C [groups * state]; the state [heads, state, head_dim] of a
    request lives at ``state[slot, state_off:]`` (float32), is read at the start of the run and left as the run
    leaves it.  ``max_run``: the longest run of the batch (None: the number of rows); long runs are cut into
    pieces that run side by side, which changes rounding only.  Returns y float32 [n, heads * head_dim]."""
    if _backend is not None:
        return _backend.ssm_scan(xbc, proj, dt_col0, dt_bias, a_log, d_skip, state, state_off, cu_seqlens, state_slots,
                                 num_requests, num_heads, head_dim, state_size, groups)
    _dev_ok(xbc, proj, dt_bias, a_log, d_skip, state, cu_seqlens, state_slots)
    inner = num_heads * head_dim
    channels = inner + 2 * groups * state_size
    if not (xbc.dtype == torch.float32 and xbc.dim() == 2 and xbc.shape[1] == channels):
        raise KernelError(f"ssm_scan: xbc must be float32 [n, {channels}]")
    n = xbc.shape[0]
    _need(proj.dtype == torch.float32 and proj.dim() == 2 and proj.shape[0] == n and 0 <= dt_col0 and dt_col0 + num_heads <= proj.shape[1],
          "ssm_scan: bad projection rows")
    for t in (dt_bias, a_log, d_skip):
        _need(t.dtype == torch.float32 and t.numel() == num_heads, "ssm_scan: per-head constants must be float32 [heads]")
    _need(state.dtype == torch.float32 and state.dim() == 2 and state.shape[1] >= state_off + num_heads * state_size * head_dim,
          "ssm_scan: state rows too short")
    _need(num_heads % groups == 0 and state_size <= 2048, "ssm_scan: heads must be a multiple of groups, state size at most 2048")
    _i32(cu_seqlens, num_requests + 1, "cu_seqlens")
    _i32(state_slots, num_requests, "state_slots")
    y = torch.empty((n, inner), dtype=torch.float32, device=xbc.device)
    max_run = n if max_run is None else min(int(max_run), n)
    lib = _Library.get()
    need = lib.tp_ssm_scan_scratch(int(num_requests), max_run, num_heads, head_dim, state_size, None)
    scratch = torch.empty((need,), dtype=torch.float32, device=xbc.device) if need else None
    _call("tp_ssm_scan", _ptr(xbc), _ptr(proj), proj.shape[1], int(dt_col0), _ptr(dt_bias), _ptr(a_log), _ptr(d_skip), _ptr(state),
          int(state.shape[1]), int(state_off), _ptr(cu_seqlens), _ptr(state_slots), _ptr(y),
          int(num_requests), num_heads, head_dim, state_size, groups, max_run, _ptr(scratch), int(need), _stream())
    return y


def gated_group_norm(y: torch.Tensor, proj: torch.Tensor, z_col0: int, weight: torch.Tensor, eps: float, groups: int,
                     out_dtype: torch.dtype) -> torch.Tensor:
    """v = y * silu(proj[:, z_col0 + j]), normed in ``groups`` equal parts (each by its own root mean square, eps
    inside the root), times ``weight``; float32 in, ``out_dtype`` [n, inner] out."""
    if _backend is not None:
        return _backend.gated_group_norm(y, proj, z_col0, weight, eps, groups, out_dtype)
    _dev_ok(y, proj, weight)
    _need(y.dtype == torch.float32 and y.dim() == 2, "gated_group_norm: y must be float32 [n, inner]")
    n, inner = y.shape
    _need(proj.dtype == torch.float32 and proj.dim() == 2 and proj.shape[0] == n and 0 <= z_col0 and z_col0 + inner <= proj.shape[1],
          "gated_group_norm: bad projection rows")
    _need(weight.dtype == torch.float32 and weight.numel() == inner and groups > 0 and inner % groups == 0, "gated_group_norm: bad weight or groups")
    out = torch.empty((n, inner), dtype=out_dtype, device=y.device)
    _call("tp_gated_group_norm", _ptr(y), _ptr(proj), proj.shape[1], int(z_col0), _ptr(weight), float(eps), _ptr(out),
          _dtcode(out_dtype), n, inner, int(groups), _stream())
    return out


def rmsnorm(h: torch.Tensor, weight: torch.Tensor, eps: float, out_dtype: torch.dtype,
            rows: Optional[torch.Tensor] = None, groups: int = 1) -> torch.Tensor:
    """float32 [n, hidden] -> out_dtype [n or len(rows), hidden].  ``groups`` > 1: the row is split into that many
    equal consecutive parts and each is divided by its own root mean square."""
    if _backend is not None:
        if groups != 1:
            return _backend.rmsnorm(h, weight, eps, out_dtype, rows, groups)
        return _backend.rmsnorm(h, weight, eps, out_dtype, rows)
    _dev_ok(h, weight, rows)
    _need(h.dtype == torch.float32 and h.dim() == 2, "rmsnorm: input must be float32 [n, hidden]")
    _need(weight.dtype == torch.float32 and weight.numel() == h.shape[1], "rmsnorm: weight must be float32 [hidden]")
    n_out = h.shape[0]
    if rows is not None:
        n_out = rows.numel()
        _i32(rows, n_out, "rmsnorm rows") if n_out else None
    out = torch.empty((n_out, h.shape[1]), dtype=out_dtype, device=h.device)
    if groups != 1:
        _need(groups > 0 and h.shape[1] % groups == 0, "rmsnorm: groups must divide the row")
        _call("tp_group_rmsnorm", _ptr(h), int(h.shape[1]), 0, _ptr(weight), _ptr(rows), _ptr(out), _dtcode(out_dtype),
              n_out, h.shape[1], int(groups), float(eps), _stream())
        return out
    _call("tp_rmsnorm", _ptr(h), _ptr(weight), _ptr(rows), _ptr(out), _dtcode(out_dtype), n_out, h.shape[1],
          float(eps), _stream())
    return out


#: bfloat16 products may use the matrix-core kernels (tests switch this off to grade the general kernel)
allow_mfma = True


def gated_layout_ok(n_rows: int, k: int) -> bool:
    """Whether ``linear_swiglu`` takes a weight of 2 * n_rows rows and k columns."""
    return n_rows % 8 == 0 and k % 32 == 0


def interleave_gate_up(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """[i, k], [i, k] -> [2i, k] with eight gate rows and eight up rows in turn, the layout
    ``linear_swiglu`` reads."""
    i, k = gate.shape
    return torch.stack([gate.reshape(i // 8, 8, k), up.reshape(i // 8, 8, k)], dim=1).reshape(2 * i, k).contiguous()


class Prenormed:
    """Rows whose root-mean-square norm is finished by the product that consumes them: ``x`` is
    bfloat16(h * norm weight) [m, k]; ``ss`` [ceil(k / 16), m] float32 (each row's values side by side in memory) holds, per block of 16 columns
    and row, the sum of squares of h; the consumer multiplies its float32 result rows by
    rsqrt(sum(ss) / k + eps).  Made by ``linear(..., residual=h, next_norm=(weight, eps))``."""
    __slots__ = ("x", "ss", "eps", "blocked")

    def __init__(self, x, ss, eps, blocked=None):
        self.x, self.ss, self.eps = x, ss, float(eps)
        #: None: ``x`` is row-major [m, k]; (m, k): ``x`` is stored k-blocked, [k / 8, m, 8] (see ``KBlocked``)
        self.blocked = blocked

    @property
    def shape(self):
        return self.x.shape if self.blocked is None else self.blocked

    def rows(self):
        """``x`` as a row-major [m, k] tensor (a copy when it is stored k-blocked)."""
        if self.blocked is None:
            return self.x
        m, k = self.blocked
        return self.x.permute(1, 0, 2).reshape(m, k)


class Unnormed:
    """float32 rows whose root-mean-square norm is left to the products that consume them: ``x`` [m, k] as it stands, the norm's
    ``weight`` [k] and ``eps`` (``norm_in_product_ok`` says for which sizes).  ``x`` must not change before they have run."""
    __slots__ = ("x", "weight", "eps")
    dtype = torch.float32

    def __init__(self, x, weight, eps):
        self.x, self.weight, self.eps = x, weight, float(eps)

    @property
    def shape(self):
        return self.x.shape


class KBlocked:
    """bfloat16 activations of at most 16 rows stored k-blocked, ``data`` [k / 8, m, 8]: eight consecutive
    columns of all rows side by side.  A product of a few rows that reads its activations straight from
    global memory then fetches neighbouring bytes instead of short pieces of several rows.  Made by
    ``linear_swiglu(..., blocked_out=True)``, taken by ``linear``."""
    __slots__ = ("data", "rows", "width")

    def __init__(self, data, rows, width):
        self.data, self.rows, self.width = data, rows, width

    @property
    def shape(self):
        return (self.rows, self.width)

    def row_major(self) -> torch.Tensor:
        return self.data.permute(1, 0, 2).reshape(self.rows, self.width).contiguous()


class TiledWeight:
    """A bfloat16 weight [n, k] (n % 16 == 0, k % 64 == 0) stored tiled, ``data`` [n / 16, k / 32, 64, 8]: the block
    of rows 16 i.. and columns 32 j.. as 1,024 contiguous bytes in the matrix cores' operand order, lane l = (column
    group l / 16, row l % 16) holding eight consecutive columns.  The products read it with whole-cache-line loads
    where the row-major form makes a wave fetch 64-byte pieces of sixteen rows.  Made by ``tile_weight``; taken by
    ``linear``, ``linear_swiglu`` and ``linear_rope_kv``."""
    __slots__ = ("data", "n", "k")

    def __init__(self, data, n, k):
        self.data, self.n, self.k = data, n, k

    @property
    def shape(self):
        return (self.n, self.k)

    @property
    def dtype(self):
        return self.data.dtype

    @property
    def device(self):
        return self.data.device

    def dim(self) -> int:
        return 2

    def rows(self, lo: int, hi: int) -> "TiledWeight":
        """Rows lo..hi (multiples of 16) as a weight of their own; no copy."""
        if not (lo % 16 == 0 and hi % 16 == 0 and 0 <= lo < hi <= self.n):
            raise KernelError(f"tiled weight: rows {lo}..{hi} of {self.n}")
        return TiledWeight(self.data[lo // 16: hi // 16], hi - lo, self.k)

    def row_major(self) -> torch.Tensor:
        """The plain [n, k] tensor (a copy)."""
        return self.data.view(self.n // 16, self.k // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(self.n, self.k).contiguous()


#: weights that fit are stored tiled (False, or TEMPURA_TILE_WEIGHTS=0 in the environment: every weight stays row-major)
tile_weights = os.environ.get("TEMPURA_TILE_WEIGHTS", "1") != "0"


def tile_weight(w: torch.Tensor):
    """A weight [n, k] for the products: ``TiledWeight`` when it is bfloat16 on the GPU with n % 16 == 0 and
    k % 64 == 0 and the matrix-core kernels are in use, else ``w`` itself.  No value changes."""
    if not (tile_weights and _backend is None and allow_mfma and isinstance(w, torch.Tensor) and w.is_cuda
            and w.dtype == torch.bfloat16 and w.dim() == 2 and w.shape[0] % 16 == 0 and w.shape[1] % 64 == 0):
        return w
    n, k = w.shape
    data = w.view(n // 16, 16, k // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous().view(n // 16, k // 32, 64, 8)
    return TiledWeight(data, n, k)


def weight_rows(w, lo: int, hi: int):
    """Rows lo..hi of a weight, tiled or not, without a copy."""
    return w.rows(lo, hi) if isinstance(w, TiledWeight) else w[lo:hi]


def _w_args(w):
    """(tensor whose memory the kernel reads, layout bit) of a weight."""
    if isinstance(w, TiledWeight):
        return w.data, 4
    return w, 0


class Partials:
    """The float32 partial sums [splits, m, n] of a product whose K was split over blocks, not yet added:
    the kernel that consumes the rows adds them (in ascending order), which saves the reduction kernel.
    Made by ``linear(..., partial_ok=True)`` and ``moe_few(..., parts)``, taken by ``rope_kv_write``, ``attention_rows`` and ``norm_add``."""
    __slots__ = ("data",)

    def __init__(self, data):
        self.data = data

    @property
    def shape(self):
        return tuple(self.data.shape[1:])


def split_norm_ok(m: int, width: int, dtype: torch.dtype) -> bool:
    """Whether the product before a norm over ``width`` columns of ``m`` rows can carry it (``linear`` with
    ``next_norm``): up to 16 rows the two products around the norm share it; with more rows the kernel that
    adds the product's partial sums into the residual stream also norms the rows, where the product splits K
    (``linear`` says whether it did)."""
    if _backend is not None:
        return _backend.split_norm_ok(m, width, dtype)
    return allow_mfma and dtype == torch.bfloat16 and 0 < m and width % 32 == 0


def _pre_args(x):
    """(the tensor a product reads, the arguments of its row scale, its rows and columns, layout bit 1 when the
    tensor is k-blocked) of plain rows or of ``Prenormed`` rows."""
    if isinstance(x, Prenormed):
        _dev_ok(x.x, x.ss.t())
        m, k = x.shape
        _need(x.x.dtype == torch.bfloat16 and x.ss.dtype == torch.float32 and x.x.numel() == m * k and
              tuple(x.ss.shape) == ((k + 15) // 16, m), "linear: malformed handed-over rows")
        return x.x, (_ptr(x.ss), x.ss.shape[0], float(x.eps)), (m, k), (1 if x.blocked is not None else 0)
    return x, (_ptr(None), 0, 0.0), (tuple(x.shape) if x.dim() == 2 else None), 0


def linear_swiglu(x, w: torch.Tensor, blocked_out: bool = False, slope: float = 1.0, limit: float = 0.0, up_offset: float = 0.0):
    """bfloat16 x [m, k] (or ``Prenormed``), interleaved gate/up weight [2i, k] -> bfloat16 [m, i] =
    silu(x g^T) * (x u^T), the gate applied to the float32 accumulators (no rounding in between).
    With ``blocked_out`` the result comes as ``KBlocked`` when there are at most 16 rows and i % 32 == 0 (else as a tensor).
    ``slope``, ``limit``, ``up_offset``: the general gate of ``gated_act`` (g' * sigmoid(slope g') * (u' + up_offset)
    with both branches limited when limit > 0) in the same epilogue (of up to 16 rows with that kernel's bits); the defaults are SwiGLU."""
    if _backend is not None:
        if (slope, limit, up_offset) != (1.0, 0.0, 0.0):
            return _backend.linear_swiglu(x, w, blocked_out, slope, limit, up_offset)
        return _backend.linear_swiglu(x, w, blocked_out) if blocked_out else _backend.linear_swiglu(x, w)
    x, pre, mk, xl = _pre_args(x)
    wd, wl = _w_args(w)
    _dev_ok(x, wd)
    if not (mk is not None and w.dim() == 2 and mk[1] == w.shape[1]):
        raise KernelError(f"linear_swiglu: shapes {mk} x {tuple(w.shape)}")
    _need(x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16, "linear_swiglu: operands must be bfloat16")
    m, k = mk
    n = w.shape[0]
    _need(n % 16 == 0 and k % 32 == 0, "linear_swiglu: needs 2i % 16 == 0 and k % 32 == 0")
    # (the product that takes such rows is an MFMA kernel over K in steps of 32)
    blocked_out = blocked_out and allow_mfma and 0 < m <= 16 and (n // 2) % 32 == 0
    if blocked_out:
        out = KBlocked(torch.empty((n // 16, m, 8), dtype=torch.bfloat16, device=x.device), m, n // 2)
    else:
        out = torch.empty((m, n // 2), dtype=torch.bfloat16, device=x.device)
    scratch, nscratch = _splitk_scratch(x, m, n)
    _call("tp_linear_fused", _ptr(x), _ptr(wd), _BF16, _ptr(out.data if blocked_out else out), _BF16, 2, m, n, k, 1,
          _ptr(scratch), int(nscratch), *pre, _ptr(None), _ptr(None), _ptr(None), (2 if blocked_out else 0) | wl | xl,
          0, _ptr(None), float(slope), float(limit), float(up_offset), 0, _ptr(None), _stream(), tag=(m, n, k))
    return out


def linear_relu2_ok(act_cols: int, k: int, dtype: torch.dtype) -> bool:
    """Whether ``linear_relu2`` takes a weight of k columns whose first ``act_cols`` rows are the activated ones."""
    return allow_mfma and dtype == torch.bfloat16 and k % 64 == 0 and act_cols % 128 == 0


def linear_act_ok(m: int, act_cols: int, k: int, dtype: torch.dtype) -> bool:
    """Whether ``linear_relu2`` takes ``m`` rows with another activation than the squared ReLU: the products of at most 16 rows."""
    return _backend is None and 0 < m <= 16 and linear_relu2_ok(act_cols, k, dtype)


def linear_relu2(x: torch.Tensor, w, act_cols: int, blocked_out: bool = False, kind: str = "relu2"):
    """bfloat16 x [m, k], weight [n, k] -> (bfloat16 [m, act_cols] = max(x w^T, 0)^2 of the first ``act_cols`` columns, the
    activation applied to the float32 accumulators; float32 [m, n - act_cols], the other columns as they are).  With
    ``blocked_out`` the first comes as ``KBlocked`` when there are at most 16 rows.  Sizes: ``linear_relu2_ok``.
    ``kind``: another of ``ACTIVATIONS`` in its place (``linear_act_ok``)."""
    if _backend is not None:
        return _backend.linear_relu2(x, w, act_cols, blocked_out)
    _need(kind == "relu2" or linear_act_ok(tuple(x.shape)[0], act_cols, tuple(x.shape)[1], torch.bfloat16), "linear_relu2: another activation takes at most 16 rows")
    wd, wl = _w_args(w)
    shape, xl = tuple(x.shape), 0
    if isinstance(x, KBlocked):
        _need(x.rows <= 16 and tuple(x.data.shape) == (x.width // 8, x.rows, 8), "linear_relu2: malformed k-blocked rows")
        x, xl = x.data, 1
    _dev_ok(x, wd)
    if not (len(shape) == 2 and w.dim() == 2 and shape[1] == w.shape[1]):
        raise KernelError(f"linear_relu2: shapes {shape} x {tuple(w.shape)}")
    _need(x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and linear_relu2_ok(act_cols, shape[1], x.dtype)
          and 0 < act_cols <= w.shape[0], "linear_relu2: needs bfloat16 operands, k % 64 == 0 and a multiple of 128 activated columns")
    (m, k), n = shape, w.shape[0]
    blocked_out = blocked_out and 0 < m <= 16
    if blocked_out:
        out = KBlocked(torch.empty((act_cols // 8, m, 8), dtype=torch.bfloat16, device=x.device), m, act_cols)
    else:
        out = torch.empty((m, act_cols), dtype=torch.bfloat16, device=x.device)
    side = torch.empty((m, n - act_cols), dtype=torch.float32, device=x.device)
    scratch, nscratch = _splitk_scratch(x, m, n)
    _call("tp_linear_fused", _ptr(x), _ptr(wd), _BF16, _ptr(out.data if blocked_out else out), _BF16, 3, m, n, k, 1, _ptr(scratch),
          int(nscratch), _ptr(None), 0, 0.0, _ptr(None), _ptr(None), _ptr(None),
          (2 if blocked_out else 0) | wl | xl | ((0 if kind == "relu2" else ACTIVATIONS[kind] + 1) << 8), 0, _ptr(None), 1.0, 0.0, 0.0, int(act_cols), _ptr(side), _stream(), tag=(m, n, k))
    return out, side


def _splitk_scratch(x: torch.Tensor, m: int, n: int):
    """Room for the partial sums of a bfloat16 product whose K is split over blocks: products of 17..128
    rows (64-row blocks up to 64 rows, 128-row blocks above), and larger ones with too few result tiles (256 x 128)
    to give every CU work."""
    if x.dtype != torch.bfloat16 or m <= 16:
        return None, 0
    if m <= 128:
        splits = min(16, max(1, -(-512 // (-(-n // 128) * -(-m // 64)))))
    else:
        tiles = -(-m // 256) * -(-n // 128)
        if tiles >= 128:
            return None, 0
        splits = min(16, 2 * -(-256 // tiles))      # (room for the library to choose: it prices the candidates)
    count = splits * m * n
    return torch.empty((count,), dtype=torch.float32, device=x.device), count


def norm_in_product_ok(x: torch.Tensor, dtype: torch.dtype) -> bool:
    """Whether the products behind a norm of the rows ``x`` may norm them themselves (``Unnormed``)."""
    # (float32, all rows that the product reading each weight once takes, so that a row's bits do not depend on the rows beside it.
    # 5,120 x 3,072, a captured chain, norm and product apart / together: 1 row 14.8 / 12.7 us, 4 rows 17.4 / 15.6, 16 rows 28.4 / 27.3)
    return _backend is None and allow_mfma and dtype == x.dtype == torch.float32 and x.dim() == 2 and 0 < x.shape[0] <= 16 and \
        x.shape[1] % 4 == 0 and x.data_ptr() % 16 == 0 and x.is_contiguous()


def linear_gate_f32_ok(x, w) -> bool:
    """Whether ``linear_gate_f32`` takes the rows ``x`` and the weight ``w`` [gate; up]."""
    return _backend is None and allow_mfma and isinstance(w, torch.Tensor) and x.dtype == w.dtype == torch.float32 and \
        0 < x.shape[0] <= 16 and x.shape[1] % 4 == 0 and w.shape[0] % 2 == 0 and w.data_ptr() % 16 == 0 and \
        (isinstance(x, Unnormed) or (x.data_ptr() % 16 == 0 and x.is_contiguous()))


def _f32_rows(x, w: torch.Tensor, gate: bool) -> torch.Tensor:
    rows, weight, eps = (x.x, x.weight, x.eps) if isinstance(x, Unnormed) else (x, None, 0.0)
    _dev_ok(rows, weight, w)
    (m, k), n = rows.shape, w.shape[0] // (2 if gate else 1)
    if not (w.dim() == 2 and w.shape[1] == k and w.dtype == torch.float32):
        raise KernelError(f"linear: shapes {(m, k)} x {tuple(w.shape)}")
    _need(weight is None or (weight.dtype == torch.float32 and weight.numel() == k), "linear: norm weight must be float32 [k]")
    out = torch.empty((m, n), dtype=torch.float32, device=rows.device)
    _call("tp_linear_f32_rows", _ptr(rows), _ptr(w), _ptr(out), m, n, k, _ptr(weight), float(eps), int(gate), _stream(),
          tag=(m, w.shape[0], k))
    return out


def linear_gate_f32(x, w: torch.Tensor) -> torch.Tensor:
    """float32 x [m, k] (or ``Unnormed``), weight [2 i, k] of gate rows and then up rows -> float32 [m, i] = silu(x g^T) * (x u^T):
    ``swiglu`` of ``linear`` in one launch for at most 16 rows (``linear_gate_f32_ok``)."""
    _need(linear_gate_f32_ok(x, w), "linear_gate_f32: needs float32 operands of at most 16 rows")
    return _f32_rows(x, w, True)


class StreamClose:
    """In the place of ``linear``'s residual: the product is a sublayer's output that closes the sublayer over ``streams`` copies of the
    stream (``stream_step``: h, mix, out_coef); with ``opening`` = (in_coef, norm weight, eps) it also opens the next one, and ``linear``
    returns that one's rows (``Prenormed`` where the product does it all, see ``stream_linear_ok``), else None."""
    __slots__ = ("h", "streams", "mix", "out_coef", "opening")

    def __init__(self, h, streams, mix, out_coef, opening=None):
        self.h, self.streams, self.mix, self.out_coef, self.opening = h, streams, mix, out_coef, opening


def stream_linear_ok(m: int, width: int, streams: int, dtype: torch.dtype) -> bool:
    """Whether a product of ``m`` rows closes a sublayer over the copies itself: few rows (one tile of the matrix cores) and four copies."""
    # (The kernel is written for four copies.  The rows go on rounded in front of the norm's scale instead of behind it, one rounding to bfloat16
    # either way.  Against 64 bits: 24 small models of four copies, 2-norm 0.0064 in front and 0.0065 behind, largest difference 0.016 and
    # 0.016 on average, from 0.006 to 0.09 by model; 4 seeds of mifutar at 4,096 0.00278 and 0.00278.  Two copies came out alike as well, but
    # one model of two copies that a test holds to a largest difference of 0.05 went from 0.030 to 0.054, which is no more than that measure
    # moves by rounding alone; so two copies keep the closing kernel.  Three and more than four were not measured.)
    return _backend is None and allow_mfma and dtype == torch.bfloat16 and 0 < m <= 16 and width % 32 == 0 and streams == 4


def _stream_linear(x, w, close: StreamClose):
    m, k = x.shape
    n, h = w.shape[0], close.h
    blocked = isinstance(x, KBlocked)
    if not (isinstance(w, TiledWeight) and stream_linear_ok(m, n, close.streams, w.dtype) and (blocked or (x.dtype == torch.bfloat16 and x.is_contiguous()))):
        y = linear(x, w, torch.float32)
        inc, weight, eps = close.opening or (None, None, 0.0)
        return stream_step(h, close.streams, y, close.mix, close.out_coef, inc, weight, eps, None if weight is None else w.dtype)
    data = x.data if blocked else x
    _dev_ok(data, w.data, h, close.mix, close.out_coef)
    if not (k == w.shape[1] and (not blocked or tuple(data.shape) == (k // 8, m, 8))):
        raise KernelError(f"linear: shapes {(m, k)} x {tuple(w.shape)}")
    _need(h.dtype == torch.float32 and tuple(h.shape) == (m, close.streams * n), "linear: the stream must be float32 [m, streams * n]")
    s = close.streams
    inc, weight, eps = close.opening or (None, None, 0.0)
    for t, size in ((close.mix, s * s), (close.out_coef, s), (inc, s), (weight, n)):
        if t is not None:
            _dev_ok(t)
            _need(t.dtype == torch.float32 and t.numel() == size, "linear: malformed coefficients of the streams")
    handed = None
    if weight is not None:
        handed = Prenormed(torch.empty((n // 8, m, 8), dtype=torch.bfloat16, device=h.device),
                           torch.empty((m, n // 16), dtype=torch.float32, device=h.device).t(), eps, (m, n))
    _call("tp_stream_linear", _ptr(data), int(blocked), _ptr(w.data), _ptr(h), s, _ptr(close.mix), _ptr(close.out_coef), _ptr(inc),
          _ptr(weight), _ptr(None if handed is None else handed.x), _ptr(None if handed is None else handed.ss), m, n, k, _stream(), tag=(m, n, k))
    return handed


def few_splits(m: int, n: int, k: int) -> int:
    """Into how many parts the K of a product of ``m`` <= 16 rows onto ``n`` columns is cut where its consumer adds partial sums: until
    there are 256 blocks of 16 columns."""
    # (from 4,096 of K on, 9.3 / 8.5 us at 2,048 columns; a shorter one is a single trip to memory for every wave anyway.  Each part a multiple
    # of 2,048, which all eight waves of a block walk in the same number of turns; other K were not measured and stay whole)
    splits = 1
    while allow_mfma and 0 < m <= 16 and k >= 4096 and splits < 4 and 2 * splits * (n // 16) <= 256 and k % (2048 * splits) == 0:
        splits *= 2
    return splits


def _split_linear(x: KBlocked, w) -> "Partials":
    m, (n, k) = x.rows, w.shape
    _dev_ok(x.data, w.data)
    _need(tuple(x.data.shape) == (k // 8, m, 8) and x.data.dtype == w.dtype == torch.bfloat16, "linear: malformed k-blocked rows")
    splits = few_splits(m, n, k)
    out = torch.empty((splits, m, n), dtype=torch.float32, device=x.data.device)
    _call("tp_split_linear", _ptr(x.data), _ptr(w.data), _ptr(out), m, n, k, splits, _stream(), tag=(m, n, k))
    return Partials(out)


def linear(x, w: torch.Tensor, out_dtype: torch.dtype, residual: Optional[torch.Tensor] = None, next_norm=None,
           partial_ok: bool = False):
    """x [m, k] (or ``Prenormed`` / ``KBlocked`` / ``Unnormed`` without a residual) @ w[n, k]^T -> out_dtype [m, n]; with ``residual`` (float32
    [m, n]) the product is added into it in place and it is returned.
    With ``next_norm`` = (float32 weight [n], eps) (needs ``residual``) the result is the pair (residual, rows
    for the part behind that norm): ``Prenormed`` rows up to 16 rows of bfloat16, the normed rows themselves
    from 17 rows on when the product's K was split (one kernel adds the partial sums into the residual and norms
    it), or None when the norm has to run on its own.
    ``residual`` may be a ``StreamClose``: the product goes into all copies of the stream, and the next sublayer's rows come back.
    With ``partial_ok`` (float32 output, no residual) the result may be ``Partials`` (of up to 16 rows: k-blocked ones and a tiled
    weight with few column blocks and a long K, ``few_splits``)."""
    if isinstance(residual, StreamClose):
        return _stream_linear(x, w, residual)
    if _backend is not None:
        if next_norm is not None:
            return _backend.linear(x, w, out_dtype, residual, next_norm)
        return _backend.linear(x, w, out_dtype, residual)
    layout = 0
    wd, wl = _w_args(w)
    if isinstance(x, Unnormed):
        if isinstance(w, torch.Tensor) and residual is None and next_norm is None and out_dtype == torch.float32 and w.data_ptr() % 16 == 0:
            return _f32_rows(x, w, False)
        x = rmsnorm(x.x, x.weight, x.eps, torch.float32)
    if isinstance(x, KBlocked):
        if partial_ok and residual is None and next_norm is None and out_dtype == torch.float32 and isinstance(w, TiledWeight) \
                and few_splits(x.rows, w.shape[0], w.shape[1]) > 1 and x.width == w.shape[1]:
            return _split_linear(x, w)
        _need(allow_mfma and x.data.dtype == torch.bfloat16 and tuple(x.data.shape) == (x.width // 8, x.rows, 8)
              and x.width % 32 == 0, "linear: malformed k-blocked rows")
        kb, layout = x, 1
        x, pre = x.data, (_ptr(None), 0, 0.0)
        m, k = kb.rows, kb.width
        _dev_ok(x, wd, residual)
        if not (w.dim() == 2 and w.shape[1] == k and w.dtype == torch.bfloat16):
            raise KernelError(f"linear: shapes {(m, k)} x {tuple(w.shape)}")
    else:
        x, pre, mk, layout = _pre_args(x)
        _dev_ok(x, wd, residual)
        if not (mk is not None and w.dim() == 2 and mk[1] == w.shape[1]):
            raise KernelError(f"linear: shapes {mk} x {tuple(w.shape)}")
        if not (x.dtype == w.dtype):
            raise KernelError(f"linear: operand dtypes differ ({x.dtype}, {w.dtype})")
        m, k = mk
    n = w.shape[0]
    if residual is not None:
        _need(residual.dtype == torch.float32 and tuple(residual.shape) == (m, n), "linear: residual must be float32 [m, n]")
        out, acc = residual, 1
    else:
        out, acc = torch.empty((m, n), dtype=out_dtype, device=x.device), 0
    post, handed = (_ptr(None), _ptr(None), _ptr(None)), None
    if next_norm is not None and split_norm_ok(m, n, x.dtype) and k % 32 == 0 and m <= 16:
        weight, eps = next_norm
        _dev_ok(weight)
        _need(residual is not None, "linear: next_norm needs a residual")
        _need(weight.dtype == torch.float32 and weight.numel() == n, "linear: norm weight must be float32 [n]")
        # (the rows go on k-blocked where the consumer can read them so: a product of a few rows then takes its
        # activations straight from memory as operands instead of staging them through LDS)
        hand_blocked = handoff_blocked and n % 32 == 0
        handed = Prenormed(torch.empty((n // 8, m, 8) if hand_blocked else (m, n), dtype=torch.bfloat16, device=x.device),
                           torch.empty((m, (n + 15) // 16), dtype=torch.float32, device=x.device).t(), eps,
                           (m, n) if hand_blocked else None)
        post = (_ptr(weight), _ptr(handed.x), _ptr(handed.ss))
        if hand_blocked:
            layout |= 8
    scratch, nscratch = _splitk_scratch(x, m, n) if allow_mfma else (None, 0)
    if allow_mfma and x.dtype == torch.float32 and m > 16:      # (parts of K where a float32 product has few result tiles)
        nscratch = int(library().tp_linear_f32_scratch(m, n, k))
        scratch = torch.empty((nscratch,), dtype=torch.float32, device=x.device) if nscratch else None
    # from 17 rows on: the partial sums of a split K may stay unadded for the kernel that consumes the rows
    layout |= wl
    defer = scratch is not None and x.dtype == torch.bfloat16 and 16 < m and (layout & 3) == 0 and \
        ((next_norm is not None and residual is not None and split_norm_ok(m, n, x.dtype) and n % 4 == 0 and n <= 16384) or
         (partial_ok and residual is None and out_dtype == torch.float32))
    splits = ctypes.c_int(1)
    _call("tp_linear_fused", _ptr(x), _ptr(wd), _dt(x), _ptr(out), _dt(out), acc, m, n, k, int(allow_mfma), _ptr(scratch),
          int(nscratch), *pre, *post, layout, int(defer), ctypes.byref(splits), 1.0,
          0.0, 0.0, 0, _ptr(None), _stream(), tag=(m, n, k))
    if defer and splits.value > 1:
        if next_norm is None:
            return Partials(scratch[: splits.value * m * n].view(splits.value, m, n))
        weight, eps = next_norm
        _dev_ok(weight)
        _need(weight.dtype == torch.float32 and weight.numel() == n, "linear: norm weight must be float32 [n]")
        normed = torch.empty((m, n), dtype=x.dtype, device=x.device)
        _call("tp_splitk_add_rmsnorm", _ptr(scratch), splits.value, _ptr(residual), _ptr(weight), float(eps),
              _ptr(normed), _dt(normed), m, n, _stream())
        return out, normed
    return out if next_norm is None else (out, handed)


#: rows handed from one product to the next with a norm between them travel k-blocked (up to 16 rows)
handoff_blocked = True
#: long steps may rotate and store in the projection's epilogue too (False: only the few rows of decoding)
rope_in_long_products = True


def linear_rope_ok(m: int, n: int, k: int, head_dim: int, rotary_dim: int, page_size: int, x_dtype: torch.dtype,
                   cache_dtype: torch.dtype, prenormed: bool = False) -> bool:
    """Whether ``linear_rope_kv`` takes a projection of m rows onto n columns: a few rows (decoding), or a long
    step with enough result tiles (128 x 128) to give half the CUs work without splitting K, heads of a multiple of 64."""
    if not (_backend is None and allow_mfma and x_dtype == torch.bfloat16 and cache_dtype == torch.bfloat16):
        return False
    if 0 < m <= 16:
        return k % 32 == 0 and head_dim % 16 == 0
    tiles = -(-m // 128) * -(-n // 128)      # (of 128 x 128, the smallest blocks of the pipelined products)
    return (rope_in_long_products and m > 128 and tiles >= 128 and k % 64 == 0 and 255 * k * 2 + 128 < 2 ** 31 and head_dim % 64 == 0
            and rotary_dim % 8 == 0 and page_size % 8 == 0 and not prenormed)


def linear_rope_kv(x, w: torch.Tensor, positions: torch.Tensor, slots: torch.Tensor, inv_freq: Optional[torch.Tensor],
                   rotary_dim: int, factor: float, num_heads: int, num_kv_heads: int, head_dim: int,
                   k_cache: torch.Tensor, v_cache: torch.Tensor, cos_sin: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The q/k/v projection of bfloat16 rows (at most 16, also ``Prenormed``; or a long step, see
    ``linear_rope_ok``) with the rotation and the cache write in its epilogue: the same result as ``linear``
    to float32 followed by ``rope_kv_write`` (w's q and k heads in paired order), without the kernel and the
    rows in between.  Returns q as bfloat16 [m, heads, head_dim]."""
    x, pre, mk, xl = _pre_args(x)
    wd, wl = _w_args(w)
    _dev_ok(x, wd, positions, slots, inv_freq, k_cache, v_cache)
    if not (mk is not None and w.dim() == 2 and mk[1] == w.shape[1]):
        raise KernelError(f"linear_rope_kv: shapes {mk} x {tuple(w.shape)}")
    m, k = mk
    n = w.shape[0]
    _need(linear_rope_ok(m, n, k, head_dim, rotary_dim, k_cache.shape[2] if k_cache.dim() == 4 else 0, x.dtype, k_cache.dtype,
                         pre[1] != 0) and w.dtype == torch.bfloat16,
          "linear_rope_kv: sizes or dtypes that the fused projection does not take (see linear_rope_ok)")
    _need(m <= 16 or cos_sin is not None, "linear_rope_kv: a long step needs the table of cosines and sines")
    if not (n == (num_heads + 2 * num_kv_heads) * head_dim):
        raise KernelError(f"linear_rope_kv: {n} weight rows for {num_heads} + 2 x {num_kv_heads} heads of {head_dim}")
    _i32(positions, m, "positions")
    _i32(slots, m, "slots")
    _need(k_cache.dim() == 4 and v_cache.dim() == 4 and k_cache.shape[1] == num_kv_heads and k_cache.shape[3] == head_dim
          and tuple(v_cache.shape) == (k_cache.shape[0], k_cache.shape[1], k_cache.shape[3], k_cache.shape[2])
          and v_cache.dtype == torch.bfloat16,
          "linear_rope_kv: caches must be k [pages, kv_heads, page_size, head_dim], v [pages, kv_heads, head_dim, page_size]")
    if rotary_dim:
        _need(inv_freq is not None and inv_freq.dtype == torch.float64 and inv_freq.numel() == rotary_dim // 2,
              "linear_rope_kv: inv_freq must be float64 [rotary_dim / 2]")
    if cos_sin is not None:
        _dev_ok(cos_sin)
        _need(cos_sin.dtype == torch.float32 and cos_sin.is_contiguous() and tuple(cos_sin.shape) == (m, rotary_dim // 2, 2),
              "linear_rope_kv: table must be float32 [m, rotary_dim / 2, 2]")
    q = torch.empty((m, num_heads, head_dim), dtype=torch.bfloat16, device=x.device)
    _call("tp_linear_rope", _ptr(x), _ptr(wd), int(wl != 0) | (2 if xl else 0), m, n, k, *pre, _ptr(positions), _ptr(slots), _ptr(inv_freq), rotary_dim,
          float(factor), num_heads, num_kv_heads, head_dim, _ptr(q), _ptr(k_cache), _ptr(v_cache),
          k_cache.shape[2], _ptr(cos_sin), _stream(), tag=(m, n, k))
    return q


def rope_kv_write(qkv, positions: torch.Tensor, slots: Optional[torch.Tensor],
                  inv_freq: Optional[torch.Tensor], rotary_dim: int, factor: float, num_heads: int,
                  num_kv_heads: int, head_dim: int, k_cache: Optional[torch.Tensor],
                  v_cache: Optional[torch.Tensor], q_dtype: torch.dtype,
                  cos_sin: Optional[torch.Tensor] = None, value_dim: Optional[int] = None,
                  pad_dim: Optional[int] = None) -> torch.Tensor:
    """Rotate q and k of float32 rows [n, (heads + 2 kv_heads) * head_dim] (or the ``Partials`` of the
    projection that makes them), store k and v into the cache rows ``slots`` and return q as q_dtype
    [n, heads, head_dim].  With ``slots`` None the rows hold q only and nothing is stored.
    ``value_dim``: the size of a value head when it is not head_dim (the rows are then
    [n, (heads + kv_heads) * head_dim + kv_heads * value_dim], the value cache [pages, kv_heads, value_dim, page_size]).
    ``pad_dim`` (>= head_dim): q comes back as [n, heads, pad_dim] and the key cache has heads of pad_dim, zeros
    behind each head's own elements (scores are unchanged; attention kernels that want keys as wide as values then serve).
    The q and k heads are in PAIRED order: elements (2 d, 2 d + 1) of a head rotate together by the angle
    of pair d (they are elements (d, d + rotary_dim / 2) of the split-half order).
    ``cos_sin``: this step's table from ``rope_table`` (the same values, computed once for all layers)."""
    vd = head_dim if value_dim is None else int(value_dim)
    od = head_dim if pad_dim is None else int(pad_dim)
    if _backend is not None:
        if vd != head_dim or od != head_dim:
            return _backend.rope_kv_write(qkv, positions, slots, inv_freq, rotary_dim, factor, num_heads,
                                          num_kv_heads, head_dim, k_cache, v_cache, q_dtype, value_dim=vd, pad_dim=od)
        return _backend.rope_kv_write(qkv, positions, slots, inv_freq, rotary_dim, factor, num_heads,
                                      num_kv_heads, head_dim, k_cache, v_cache, q_dtype)
    splits = 1
    if isinstance(qkv, Partials):
        splits, qkv = qkv.data.shape[0], qkv.data.view(-1, qkv.data.shape[2])[: qkv.data.shape[1]]
        _need(qkv.is_contiguous() or splits == 1, "rope_kv_write: malformed partial sums")
    _dev_ok(positions, slots, inv_freq, k_cache, v_cache)
    _need(qkv.is_cuda, "operand is not on the GPU")
    _need(qkv.dtype == torch.float32 and qkv.dim() == 2, "rope_kv_write: rows must be float32 [n, width]")
    n = qkv.shape[0]
    width = (num_heads + (num_kv_heads if slots is not None else 0)) * head_dim + (num_kv_heads * vd if slots is not None else 0)
    if not (qkv.shape[1] == width):
        raise KernelError(f"rope_kv_write: row width {qkv.shape[1]} != {width}")
    _i32(positions, n, "positions") if n else None
    page_size, cache_dt = 1, _F32
    if slots is not None:
        _i32(slots, n, "slots") if n else None
        _need(k_cache is not None and v_cache is not None and k_cache.dim() == 4 and v_cache.dim() == 4
              and tuple(v_cache.shape) == (k_cache.shape[0], k_cache.shape[1], vd, k_cache.shape[2]),
              "rope_kv_write: caches must be k [pages, kv_heads, page_size, head_dim], v [pages, kv_heads, value_dim, page_size]")
        _need(k_cache.shape[1] == num_kv_heads and k_cache.shape[3] == od, "rope_kv_write: cache layout mismatch")
        _need(k_cache.dtype == v_cache.dtype, "rope_kv_write: cache dtypes differ")
        page_size, cache_dt = k_cache.shape[2], _dt(k_cache)
    if rotary_dim:
        _need(inv_freq is not None and inv_freq.dtype == torch.float64 and inv_freq.numel() == rotary_dim // 2,
              "rope_kv_write: inv_freq must be float64 [rotary_dim / 2]")
    if cos_sin is not None:
        _need(cos_sin.is_cuda and cos_sin.dtype == torch.float32 and cos_sin.is_contiguous()
              and tuple(cos_sin.shape) == (n, rotary_dim // 2, 2), "rope_kv_write: table must be float32 [n, rotary_dim / 2, 2]")
    _need(od >= head_dim and od % 2 == 0, "rope_kv_write: pad_dim must be even and at least head_dim")
    q = torch.empty((n, num_heads, od), dtype=q_dtype, device=qkv.device)
    _call("tp_rope_kv_write", _ptr(qkv), qkv.shape[1], _ptr(positions), _ptr(slots), _ptr(inv_freq), rotary_dim,
          float(factor), n, num_heads, num_kv_heads, head_dim, _ptr(q), _dtcode(q_dtype),
          _ptr(k_cache), _ptr(v_cache), cache_dt, page_size, splits, _ptr(cos_sin), vd, od, _stream())
    return q


def rope_table(positions: torch.Tensor, inv_freq: torch.Tensor, rotary_dim: int, factor: float) -> torch.Tensor:
    """float32 [n, rotary_dim / 2, 2]: cosine and sine (times factor) of every token's angles, as
    ``rope_kv_write`` would compute them itself."""
    if _backend is not None:
        return None
    _dev_ok(positions, inv_freq)
    n = positions.numel()
    _i32(positions, n, "positions") if n else None
    _need(rotary_dim > 0 and inv_freq.dtype == torch.float64 and inv_freq.numel() == rotary_dim // 2,
          "rope_table: inv_freq must be float64 [rotary_dim / 2]")
    table = torch.empty((n, rotary_dim // 2, 2), dtype=torch.float32, device=positions.device)
    _call("tp_rope_table", _ptr(positions), _ptr(inv_freq), rotary_dim, float(factor), n, _ptr(table), _stream())
    return table


#: bfloat16 attention may use the matrix-core kernels
allow_fast_attention = True
#: the split decode kernel aims at this many blocks (of four waves) in flight
decode_target_blocks = 256


def decode_rows_padded(rows: int) -> int:
    """The number of rows a decode step of `rows` requests is sized for: the next power of two up to 128, beyond
    that the next multiple of 128.  A captured step has that many rows and an eager one chooses its kernels and
    splits as if it had, so the two give the same bits."""
    if rows > 128:
        return (rows + 127) // 128 * 128
    padded = 1
    while padded < rows:
        padded *= 2
    return padded
#: and at least this many splits while a split has at most 64 blocks
decode_min_splits = 8
#: measurements: this many splits whatever the batch (0: chosen by the rules below)
decode_force_splits = 0
#: steps of single tokens take their attention from the projection's rows where its kernel allows it
rows_attention = True
#: portions of prompts with fewer query blocks than this have their keys split over blocks (1: never)
portion_target_blocks = 1024
#: in parts of at least this many keys
portion_min_keys = 1024
#: and only while the partial results stay below this many bytes
portion_scratch_limit = 256 << 20


#: the pairs (key size, value size) the matrix-core attention kernels are built for
FAST_PAIRS = ((32, 32), (64, 64), (96, 96), (128, 128), (64, 32), (128, 64), (160, 96), (192, 128), (288, 256), (320, 256), (576, 512))


def fast_pair(key_dim: int, value_dim: int, exact_values: bool = True):
    """The smallest pair of ``FAST_PAIRS`` whose key size is at least ``key_dim`` and whose value size is ``value_dim``
    (``exact_values`` False: at least ``value_dim``), or None.  A part pads its keys (values) with zeros up to it."""
    fit = [p for p in FAST_PAIRS if p[0] >= key_dim and (p[1] == value_dim if exact_values else p[1] >= value_dim)]
    return min(fit, key=lambda p: (p[0] + p[1], p)) if fit else None


def decode_rings(key_dim: int, value_dim: int, page_size: int) -> bool:
    """Whether single tokens take the kernel whose waves have their keys and values on the way to LDS."""
    return key_dim in (32, 64, 128, 192) and (key_dim + value_dim) % 64 == 0 and value_dim <= 128 and page_size >= 16 and page_size & (page_size - 1) == 0


def fast_attention_takes(has_sink: bool, keep_first: int) -> bool:
    """Whether the matrix-core attention kernels take a softmax with a sink and kept first keys (else the general
    kernel runs, and no splits or partial results are prepared for them): both (kept first keys by the kernels that
    load keys and values per wave, whose portions are never split over blocks)."""
    return True


def _keys_seen(max_context_len: int, window: int, keep_first: int, chunk: int) -> int:
    """The most keys that a single token sees, by the longest context rounded up to a power of two from 256: a step captured for a bound on
    the context and an eager step at the actual length then decide alike and give the same bits."""
    bound = 256
    while bound < max_context_len:
        bound *= 2
    return min(bound, window + keep_first + 31) if window else min(bound, chunk) if chunk else bound


def _decode_splits(requests: int, heads: int, kvh: int, max_context_len: int, window: int, keep_first: int, chunk: int, rings: bool) -> int:
    """Into how many splits the keys of a step's single tokens are cut (``rings``: by the kernel of ``decode_rings``)."""
    # enough blocks to fill 256 CUs, but at least 128 keys per block
    blocks_per_split = decode_rows_padded(requests) * kvh * ((heads // kvh + 15) // 16)
    # (two blocks fit a CU, 512 the chip.  From 65 to 256 blocks per split, as many splits as fill it once: measured
    # alone at 2,100 keys, 16 requests 35.8 -> 33.5 us, 20 requests 47.2 -> 38.5, 32 requests 54.3 -> 52.7, and more
    # for contexts that differ; through the engine 16 requests of the 8B shape 4.33 -> 4.25 ms a step, 32 requests
    # 5.27 -> 5.20; 12 requests in five splits against three 4.11 / 4.27, 20 in three against two 4.77 / 4.92, 24 in
    # two against three 4.97 / 5.21.)
    if blocks_per_split <= 64:
        want = -(-decode_target_blocks // blocks_per_split)
    elif blocks_per_split <= decode_target_blocks:
        want = max(1, 2 * decode_target_blocks // blocks_per_split)
    else:
        # (more blocks than half the chip's places: no split.  Through the engine, requests of 2,048+ keys of the 8B
        # shape, one split against two: 36 requests 6.06 / 5.97 ms a step, 40: 6.14 / 6.04, 48: 6.27 / 6.49,
        # 56: 6.42 / 6.68, 64: 6.62 / 6.89; three splits at 36 and 40 requests, which the kernel timed alone
        # prefers, 6.07 and 6.13)
        want = 1
    if blocks_per_split <= 64:
        want = max(want, decode_min_splits)     # (batch 8 of the 8B shape: eight splits 3.87 ms a step, four 3.94)
    if decode_force_splits > 0:
        want = decode_force_splits
    seen = _keys_seen(max_context_len, window, keep_first, chunk)      # (at least 128 keys a split)
    if decode_force_splits == 0 and rings:
        # (a launch and a trip through memory for the kernel that adds the splits, 4 us, against the keys that one block walks
        # alone, 5 us for 512 of 128 elements: 8 key heads of 128, not split / as above, one request of 120 / 500 / 1,000 keys
        # 4.6 / 8.6 / 13.4 against 8.0 / 10.4 / 8.8 us, 8 requests 5.8 / 9.4 / 14.2 against 9.0 / 12.0 / 12.5.  From 65 blocks a
        # split on: 16 requests of 1,000 keys 15.8 against 19.5 us, of 3,000 41.9 against 39.8 and in two splits 38.4, of 600 to
        # 6,000 59 and 43.5; from 129 on: 32 requests of 500 / 1,000 / 3,000 keys 13.9 / 23.6 / 64 against 18.1 / 28.5 / 68,
        # of 600 to 6,000 73.8 against 82.)
        if seen <= 512 or blocks_per_split > 128:
            want = 1
        elif blocks_per_split > 64:
            want = 1 if seen <= 1024 else 2
    return max(1, min(64, want, max(1, seen // 128)))


def _decode_waves(requests: int, heads: int, kvh: int, splits: int) -> int:
    """How many waves a block of the kernel of ``decode_rings`` has: eight where the keys are not split and every block has a CU of its own,
    else four, by the rows that the step is sized for (the order of a row's sums hangs on it)."""
    # (one request of 500 keys of 64 elements 7.2 -> 6.4 us, 32 of 3,000 36.1 -> 35.6; 48 requests, 384 blocks, 20.6 -> 22.7)
    return 8 if splits == 1 and decode_rows_padded(requests) * kvh * ((heads // kvh + 15) // 16) <= 256 else 4


def decode_order(shared: Optional[dict], context_lens: torch.Tensor, n: int, heads: int, kvh: int, splits: int, window: int, keep_first: int,
                 chunk: int) -> Optional[torch.Tensor]:
    """The order of a step's single tokens among the blocks of the kernel of ``decode_rings`` (int32 [n]), or None: as they are.  ``shared``: the
    step's (``StepContext.shared``; without it no order is made): its layers with the same mask and heads share one."""
    # (one launch a step, 2.4 us, and 0.2 us a layer; up to as many blocks as CUs there is nothing to choose)
    per = kvh * ((heads // kvh + 15) // 16)
    places = 256 // per
    if shared is None or splits != 1 or not 0 < places < n <= 512 or _decode_waves(n, heads, kvh, splits) != 4:
        return None
    key = ("decode_order", n, places, int(window), int(keep_first), int(chunk))
    if key not in shared:
        _dev_ok(context_lens)
        _i32(context_lens, n, "context_lens")
        order = torch.empty((n,), dtype=torch.int32, device=context_lens.device)
        _call("tp_decode_order", _ptr(context_lens), n, int(window), int(keep_first), int(chunk), places, _ptr(order), _stream())
        shared[key] = order
    return shared[key]


def paged_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, block_tables: torch.Tensor,
                    cu_seqlens: torch.Tensor, context_lens: torch.Tensor, token_req: torch.Tensor,
                    scale: float, window: int, max_q_len: int, max_context_len: int,
                    num_single: Optional[int] = None, dist_bias: Optional[torch.Tensor] = None,
                    sink: Optional[torch.Tensor] = None, keep_first: int = 0, chunk: int = 0, softcap: float = 0.0,
                    into: Optional[tuple] = None, shared: Optional[dict] = None) -> Optional[torch.Tensor]:
    """q [n, heads, head_dim] over k [pages, kv_heads, page_size, head_dim] and transposed
    v [pages, kv_heads, value_dim, page_size] -> [n, heads * value_dim] (value_dim is the value cache's own; the
    matrix-core kernels take the pairs of sizes in ``FAST_PAIRS``, other sizes run the general kernel).
    ``dist_bias`` (float32 [heads, L]): added to the scaled score of a query at position p and a key at j as
    dist_bias[head, min(p - j, L - 1)].
    ``sink`` (float32 [heads]): the softmax's denominator holds one more term, exp(sink[head]), without key or value.
    ``keep_first``: under a window, the request's first ``keep_first`` keys stay visible as well.
    ``chunk`` (instead of a window): a query sees the keys of its own aligned chunk of that many positions only.
    ``softcap`` > 0: a scaled score s becomes softcap * tanh(s / softcap) before the softmax (no distance bias then).
    ``into``: the last six arguments of ``sigmoid_gate`` (gate rows or None, their column, scale, output rows, their column, columns
    that share a gate): the result goes there and None comes back.  ``shared``: the step's (``StepContext.shared``, see ``decode_order``)."""
    if into is not None and not (_backend is None and num_single == block_tables.shape[0] == q.shape[0]):
        sigmoid_gate(paged_attention(q, k_cache, v_cache, block_tables, cu_seqlens, context_lens, token_req, scale, window, max_q_len,
                                     max_context_len, num_single, dist_bias, sink, keep_first, chunk, softcap), *into)
        return None
    if _backend is not None:
        if chunk or softcap:
            return _backend.paged_attention(q, k_cache, v_cache, block_tables, cu_seqlens, context_lens,
                                            token_req, scale, window, max_q_len, max_context_len, dist_bias=dist_bias,
                                            sink=sink, keep_first=keep_first, chunk=chunk, softcap=softcap)
        if sink is not None or keep_first:
            return _backend.paged_attention(q, k_cache, v_cache, block_tables, cu_seqlens, context_lens,
                                            token_req, scale, window, max_q_len, max_context_len, dist_bias=dist_bias,
                                            sink=sink, keep_first=keep_first)
        if dist_bias is not None:
            return _backend.paged_attention(q, k_cache, v_cache, block_tables, cu_seqlens, context_lens,
                                            token_req, scale, window, max_q_len, max_context_len, dist_bias=dist_bias)
        return _backend.paged_attention(q, k_cache, v_cache, block_tables, cu_seqlens, context_lens,
                                        token_req, scale, window, max_q_len, max_context_len)
    # num_single: requests that bring exactly one token (None: all of them iff max_q_len == 1, else unknown
    # and every request is treated as a portion).
    _dev_ok(q, k_cache, v_cache, block_tables, cu_seqlens, context_lens, token_req)
    _need(q.dim() == 3 and k_cache.dim() == 4 and v_cache.dim() == 4, "paged_attention: bad operand ranks")
    n, heads, d = q.shape
    pages, kvh, page_size, d2 = k_cache.shape
    vd = v_cache.shape[2]
    _need(tuple(v_cache.shape) == (pages, kvh, vd, page_size), "paged_attention: v cache must be [pages, kv_heads, value_dim, page_size]")
    _need(d == d2, "paged_attention: head_dim of q and cache differ")
    _need(q.dtype == k_cache.dtype == v_cache.dtype, "paged_attention: q and cache dtypes differ")
    _need(block_tables.dim() == 2 and block_tables.dtype == torch.int32, "paged_attention: block_tables must be int32 [r, width]")
    r, width = block_tables.shape
    _i32(cu_seqlens, r + 1, "cu_seqlens")
    _i32(context_lens, r, "context_lens")
    _i32(token_req, n, "token_req") if n else None
    _need(pages * kvh * page_size < 2 ** 31, "paged_attention: cache pool too large for 32-bit row indices")
    _need(max_context_len <= width * page_size, "paged_attention: block table narrower than the longest context")
    if num_single is None:
        num_single = r if max_q_len == 1 else 0
    _need(0 <= num_single <= r, "paged_attention: num_single out of range")
    if dist_bias is not None:
        _dev_ok(dist_bias)
        _need(dist_bias.dtype == torch.float32 and dist_bias.dim() == 2 and dist_bias.shape[0] == heads and dist_bias.shape[1] > 0,
              "paged_attention: dist_bias must be float32 [heads, L]")
    if sink is not None:
        _dev_ok(sink)
        _need(sink.dtype == torch.float32 and sink.numel() == heads, "paged_attention: sink must be float32 [heads]")
    _need(keep_first >= 0, "paged_attention: keep_first must be >= 0")
    _need(chunk >= 0 and not (chunk and window), "paged_attention: chunks and a window exclude each other")
    _need(softcap >= 0 and not (softcap and dist_bias is not None), "paged_attention: a cap and a distance bias exclude each other")
    if chunk == 1:      # (a chunk of one position: the query itself)
        chunk, window = 0, 1
    if not window:
        keep_first = 0
    fast = allow_fast_attention and q.dtype == torch.bfloat16 and (d, vd) in FAST_PAIRS and page_size % 8 == 0
    fast = fast and (dist_bias is None or d == vd)
    fast = fast and fast_attention_takes(sink is not None, keep_first) and not (keep_first and dist_bias is not None)
    splits, scratch, order = 1, None, None
    if fast and num_single > 0:
        splits = _decode_splits(num_single, heads, kvh, max_context_len, window, keep_first, chunk, dist_bias is None and decode_rings(d, vd, page_size))
        if splits > 1:
            scratch = torch.empty((r * heads * splits * (vd + 2),), dtype=torch.float32, device=q.device)
        if num_single == r == n and dist_bias is None and decode_rings(d, vd, page_size):
            order = decode_order(shared, context_lens, n, heads, kvh, splits, window, keep_first, chunk)
    fast_f32 = allow_fast_attention and q.dtype == torch.float32 and d == vd and d in (32, 64, 96, 128) and page_size % 16 == 0
    if fast_f32 and max_q_len == 1 and n == r:
        # (float32: at least 128 keys a block of four waves, by the same bound on the context as above, until there are
        # two blocks a CU)
        bound = 256
        while bound < max_context_len:
            bound *= 2
        splits = max(1, min(64, bound // 128, 512 // (decode_rows_padded(r) * kvh)))
        if splits > 1:
            scratch = torch.empty((r * heads * splits * (vd + 2),), dtype=torch.float32, device=q.device)
    parts, part_scratch = 1, None
    # (the kernel with a distance bias does not split a portion's keys)
    if fast and dist_bias is None and not keep_first and num_single < r and d in (32, 64, 128, 192) and (d + vd) % 64 == 0 and page_size & (page_size - 1) == 0 and page_size >= max(8, 512 // d):
        # Few query blocks under a long context (a portion of a prompt behind a long cached prefix): the keys of
        # every portion are split over blocks until the chip is full (T = 512 behind 7,680 keys: 219 -> 137 us).
        q_blocks = -(-(n - num_single) // 32) + (r - num_single)
        blocks = q_blocks * kvh * ((heads // kvh + 3) // 4)
        # (a query block is split into at most as many parts as it has portion_min_keys keys: the short blocks
        # of a prompt from an empty cache stay whole)
        parts = max(1, min(16, portion_target_blocks // blocks, max_context_len // portion_min_keys, 65535 // r))
        if parts > 1 and n * heads * parts * (vd + 4) * 4 > portion_scratch_limit:
            parts = 1
        if parts > 1:
            part_scratch = torch.empty((n * heads * parts * (vd + 4),), dtype=torch.float32, device=q.device)
    # (single tokens: the kernel that writes a row also gates it)
    gated = into is not None and fast and num_single == r == n and 0 < n <= 65535
    if not gated:
        gate, gate_col0, factor, dest_col0, per = None, 0, 1.0, 0, 1
        dest = torch.empty((n, heads * vd), dtype=q.dtype, device=q.device)
    else:
        gate, gate_col0, factor, dest, dest_col0, per = into
        _dev_ok(gate, dest)
        _need(dest.dim() == 2 and dest.dtype == q.dtype and dest.shape[0] == n and 0 <= dest_col0 and dest_col0 + heads * vd <= dest.shape[1]
              and per >= 1 and (heads * vd) % per == 0, "paged_attention: bad output rows")
        _need(gate is None or (gate.dtype == torch.float32 and gate.dim() == 2 and gate.shape[0] == n and 0 <= gate_col0
                               and gate_col0 + heads * vd // per <= gate.shape[1]), "paged_attention: bad gate rows")
    _call("tp_paged_attention", _ptr(q), _dt(q), _ptr(k_cache), _ptr(v_cache), _ptr(block_tables), width,
          _ptr(cu_seqlens), _ptr(context_lens), _ptr(token_req), _ptr(dest), n, r, heads, kvh, d, page_size,
          float(scale), int(window), int(max_q_len), int(max_context_len), 2 if gated else int(fast or fast_f32),
          int(num_single), int(splits), _decode_waves(max(1, num_single), heads, kvh, splits), _ptr(scratch), int(parts), max(1, portion_min_keys // 32), _ptr(part_scratch),
          _ptr(dist_bias), 0 if dist_bias is None else dist_bias.shape[1], int(vd), int(keep_first), _ptr(sink), int(chunk),
          float(softcap), _ptr(gate), 0 if gate is None else gate.shape[1], int(gate_col0), int(per), float(factor),
          dest.shape[1], int(dest_col0), _ptr(order), _stream())
    if into is None:
        return dest
    if not gated:
        sigmoid_gate(dest, *into)
    return None


def attention_rows_ok(rows, ctx, heads: int, kvh: int, dim: int, value_dim: int, k_cache: torch.Tensor, conv_taps: int = 0, window: int = 0,
                      col0: int = 0, state: Optional[torch.Tensor] = None, state_off: int = 0) -> bool:
    """Whether ``attention_rows`` takes a projection's float32 ``rows`` (or ``Partials``) from column ``col0`` on: a step of single tokens,
    bfloat16 caches, and everything read in pairs of floats at even places, the carried inputs of a convolution (from ``state_off`` on in
    the rows of ``state``) among them."""
    data = rows.data if isinstance(rows, Partials) else rows
    page_size = k_cache.shape[2]
    if not (_backend is None and allow_fast_attention and rows_attention and k_cache.dtype == torch.bfloat16 and k_cache.shape[3] == dim == value_dim
            and dim in (64, 128) and decode_rings(dim, dim, page_size) and heads // kvh <= 16 and ctx.num_requests == ctx.num_single == ctx.num_tokens
            and ctx.num_tokens <= 65535 and data.dtype == torch.float32 and data.shape[-1] % 2 == 0 and data.data_ptr() % 8 == 0 and col0 % 2 == 0
            and (data.dim() == 2 or data.shape[0] <= 8)):
        return False
    if conv_taps and state is not None and (state.shape[1] % 2 != 0 or state_off % 2 != 0 or state.data_ptr() % 8 != 0):
        return False
    # (a channel's carried inputs have one block: with a convolution the keys are not split, for which 1,024 keys are a microsecond more
    # than split, and the two launches in front of the attention 5)
    if conv_taps:
        seen = min(_keys_seen(ctx.max_context_len, 0, 0, 0), window or 1 << 30)
        return conv_taps <= 4 and data.dim() == 2 and (seen <= 1024 or decode_rows_padded(ctx.num_tokens) * kvh > 64)
    return True


def attention_rows_pays(ctx, kvh: int, dim: int, window: int = 0, keep_first: int = 0, chunk: int = 0) -> bool:
    """Whether ``attention_rows`` is the faster way where it could be taken: its blocks work their rows out before they begin with their keys."""
    # (A launch of 4 to 5 us saved against that start.  Where two blocks a CU and more share a long stream of keys the start costs more: steps
    # of 32 layers, 8 key heads of 128, from rows / with the launches apart, 32 requests of 500 / 1,000 / 3,000 keys 3.82 / 3.90, 4.15 / 4.22 and
    # 5.45 / 5.50 ms, 48 of 500 / 1,800 / 3,000 4.23 / 4.27, 5.53 / 5.56 and 6.69 / 6.68, 64 of 400 / 800 / 3,000 4.25 / 4.29, 4.79 / 4.78 and
    # 7.69 / 7.53; 128 of 800 / 1,500 / 3,050 7.44 / 7.35, 9.34 / 9.13 and 13.79 / 13.49.  Heads of 64 carry half the bytes a key: the kernels
    # alone 64 of 3,000 keys 69.3 / 69.5 us, 128 of 800 / 3,000 45.6 / 48.0 and 132.8 / 135.0, with a convolution 55.9 / 57.5 and 152 / 146.)
    blocks = decode_rows_padded(ctx.num_tokens) * kvh
    return blocks <= 256 or _keys_seen(ctx.max_context_len, window, keep_first, chunk) * dim <= (2048 if blocks <= 512 else 512) * 128


def _rows_splits(ctx, heads: int, kvh: int, window: int, keep_first: int, chunk: int, conv: bool, beside: bool) -> int:
    splits = 1 if conv else _decode_splits(ctx.num_tokens, heads, kvh, ctx.max_context_len, window, keep_first, chunk, True)
    return -(-splits // 2) if beside else splits        # (blocks of eight waves instead of four)


def attention_beside_ok(ctx, heads: int, kvh: int, window: int, conv_taps: int, step_heads: int) -> bool:
    """Whether ``attention_rows`` should run a recurrent mixer's step in its launch: while the blocks of both have a CU each."""
    # (of the rows that the step is sized for: beside the mixer the keys are cut otherwise, and a captured step has to do as an eager one)
    return decode_rows_padded(ctx.num_tokens) * (kvh * _rows_splits(ctx, heads, kvh, window, 0, 0, conv_taps > 0, True) + step_heads) <= 256


def attention_rows(rows, col0: int, ctx, group: int, heads: int, kvh: int, dim: int, k_cache: torch.Tensor, v_cache: torch.Tensor, scale: float,
                   inv_freq: Optional[torch.Tensor], rotary_dim: int, factor: float, cos_sin: Optional[torch.Tensor], window: int = 0,
                   keep_first: int = 0, chunk: int = 0, sink: Optional[torch.Tensor] = None, norms=None, norm_eps: float = 0.0, conv=None,
                   into: Optional[tuple] = None, beside=None) -> Optional[torch.Tensor]:
    """A step of single tokens from their projection's rows (q | k | v from column ``col0`` on, or ``Partials``) to the heads' outputs:
    ``causal_conv`` without activation (``conv`` = (weights [taps, channels], state, its column)), a norm per head of q and k (``norms``),
    ``rope_kv_write`` and ``paged_attention`` in one launch.  ``beside``: a recurrent mixer's step of the same requests, written down by
    ``delta_step`` or ``linear_step``, which runs in that launch too.  ``ctx``: the step; ``group``: its cache group.  Sizes: ``attention_rows_ok``."""
    parts, data = 1, rows
    if isinstance(rows, Partials):
        parts, data = rows.data.shape[0], rows.data.view(-1, rows.data.shape[2])
    n, stride = ctx.num_tokens, data.shape[1]
    bt = ctx.block_tables[group]
    slots = ctx.slot_mapping[group]
    _dev_ok(data, k_cache, v_cache, bt, ctx.context_lens, ctx.positions, slots, inv_freq, cos_sin, sink)
    _need(attention_rows_ok(rows, ctx, heads, kvh, dim, v_cache.shape[2], k_cache, 0 if conv is None else conv[0].shape[0], window, col0,
                            *(() if conv is None else conv[1:])), "attention_rows: sizes that it does not take")
    _need(data.shape[0] == parts * n and col0 >= 0 and col0 + (heads + 2 * kvh) * dim <= stride, "attention_rows: bad rows")
    pages, _, page_size, _ = k_cache.shape
    _need(k_cache.shape[1] == kvh and tuple(v_cache.shape) == (pages, kvh, dim, page_size) and v_cache.dtype == torch.bfloat16, "attention_rows: bad caches")
    _need(pages * kvh * page_size < 2 ** 31, "paged_attention: cache pool too large for 32-bit row indices")
    _need(bt.dtype == torch.int32 and bt.shape[0] == n and ctx.max_context_len <= bt.shape[1] * page_size, "attention_rows: bad block table")
    _i32(ctx.context_lens, n, "context_lens")
    _i32(ctx.positions, n, "positions")
    _i32(slots, n, "slots")
    if rotary_dim:
        _need(inv_freq is not None and inv_freq.dtype == torch.float64 and inv_freq.numel() == rotary_dim // 2, "attention_rows: inv_freq must be float64 [rotary_dim / 2]")
    if cos_sin is not None:
        _need(cos_sin.dtype == torch.float32 and tuple(cos_sin.shape) == (n, rotary_dim // 2, 2), "attention_rows: table must be float32 [n, rotary_dim / 2, 2]")
    if sink is not None:
        _need(sink.dtype == torch.float32 and sink.numel() == heads, "attention_rows: sink must be float32 [heads]")
    if norms is not None:
        _dev_ok(*norms)
        _need(all(w.dtype == torch.float32 and w.numel() == dim for w in norms), "attention_rows: norm weights must be float32 [dim]")
    conv_w, state, state_off = conv if conv is not None else (None, None, 0)
    if conv is not None:
        _dev_ok(conv_w, state)
        _need(conv_w.dtype == state.dtype == torch.float32 and conv_w.dim() == state.dim() == 2 and conv_w.shape[1] == (heads + 2 * kvh) * dim,
              "attention_rows: bad convolution")
        _i32(ctx.state_slots, n, "state_slots")
    if chunk == 1:
        chunk, window = 0, 1
    splits = _rows_splits(ctx, heads, kvh, window, keep_first, chunk, conv is not None, beside is not None)
    scratch = torch.empty((n * heads * splits * (dim + 2),), dtype=torch.float32, device=data.device) if splits > 1 else None
    order = None if beside is not None else decode_order(getattr(ctx, "shared", None), ctx.context_lens, n, heads, kvh, splits, window,
                                                         keep_first if window else 0, chunk)
    if into is not None:
        gate, gate_col0, gate_scale, out, out_col0, per = into
        _dev_ok(gate, out)
        _need(out.dim() == 2 and out.dtype == torch.bfloat16 and out.shape[0] == n and 0 <= out_col0 and out_col0 + heads * dim <= out.shape[1]
              and per >= 1 and (heads * dim) % per == 0, "attention_rows: bad output rows")
        _need(gate is None or (gate.dtype == torch.float32 and gate.dim() == 2 and gate.shape[0] == n and 0 <= gate_col0
                               and gate_col0 + heads * dim // per <= gate.shape[1]), "attention_rows: bad gate rows")
    else:
        gate, gate_col0, gate_scale, out_col0, per = None, 0, 1.0, 0, 1
        out = torch.empty((n, heads * dim), dtype=torch.bfloat16, device=data.device)
    _call("tp_attention_rows", (data.data_ptr() + 4 * col0), int(n * stride), stride, parts,
          _ptr(conv_w), 0 if conv_w is None else conv_w.shape[0], 0 if conv_w is None else conv_w.shape[1], _ptr(state),
          int(0 if state is None else state.shape[1]), int(state_off), _ptr(ctx.state_slots if conv is not None else None),
          _ptr(None if norms is None else norms[0]), _ptr(None if norms is None else norms[1]), float(norm_eps), _ptr(ctx.positions),
          _ptr(inv_freq), int(rotary_dim), float(factor), _ptr(cos_sin), _ptr(slots), _ptr(k_cache), _ptr(v_cache), _ptr(bt), bt.shape[1],
          _ptr(ctx.cu_seqlens), _ptr(ctx.context_lens), _ptr(out), n, heads, kvh, dim, page_size, float(scale), int(window), int(keep_first),
          int(chunk), _ptr(sink), int(splits), 8 if beside is not None else _decode_waves(n, heads, kvh, splits), _ptr(scratch), int(into is not None), _ptr(gate), 0 if gate is None else gate.shape[1], int(gate_col0),
          int(per), float(gate_scale), out.shape[1], int(out_col0), beside, _ptr(order), _stream())
    return None if into is not None else out


def swiglu(gu: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """[m, 2i] (gate columns then up columns) -> out_dtype [m, i]."""
    if _backend is not None:
        return _backend.swiglu(gu, out_dtype)
    _dev_ok(gu)
    _need(gu.dim() == 2 and gu.shape[1] % 2 == 0, "swiglu: input must be [m, 2i]")
    m, i2 = gu.shape
    out = torch.empty((m, i2 // 2), dtype=out_dtype, device=gu.device)
    _call("tp_swiglu", _ptr(gu), _dt(gu), _ptr(out), _dtcode(out_dtype), m, i2 // 2, _stream())
    return out


def argmax(logits: torch.Tensor) -> torch.Tensor:
    """float32 [m, vocab] -> int32 [m]; the last maximum wins on exact ties."""
    if _backend is not None:
        return _backend.argmax(logits)
    _dev_ok(logits)
    _need(logits.dtype == torch.float32 and logits.dim() == 2, "argmax: logits must be float32 [m, vocab]")
    out = torch.empty((logits.shape[0],), dtype=torch.int32, device=logits.device)
    part = torch.empty((logits.shape[0] * 128,), dtype=torch.float32, device=logits.device)
    _call("tp_argmax", _ptr(logits), _ptr(out), logits.shape[0], logits.shape[1], _ptr(part), _stream())
    return out


class HostCopy:
    """A small device tensor on its way to the host: the copy into pinned memory is queued when the object is
    made, ``result()`` waits for that copy alone (not for work queued behind it) and returns a list.  The pinned
    buffers are taken in turn from a ring, so at most ``RING`` copies may be outstanding."""
    RING = 8
    _ring: list = []
    _next = 0

    def __init__(self, t: torch.Tensor):
        cls = HostCopy
        n = t.numel()
        if not cls._ring:
            cls._ring = [None] * cls.RING
        slot = cls._ring[cls._next]
        if slot is None or slot[0].numel() < n or slot[0].dtype != t.dtype:
            slot = (torch.empty(max(n, 256), dtype=t.dtype, pin_memory=True), torch.cuda.Event())
            cls._ring[cls._next] = slot
        cls._next = (cls._next + 1) % cls.RING
        self._buf, self._event, self._n = slot[0], slot[1], n
        self._buf[:n].copy_(t.reshape(-1), non_blocking=True)
        self._event.record()

    def result(self) -> list:
        self._event.synchronize()
        return self._buf[: self._n].tolist()


class _Staging:
    """Small per-call option arrays on their way to the device through pinned memory: the copy is queued behind
    the work in flight instead of making the host wait for it (a pageable copy would).  Buffers are taken in
    turn from a ring and reused once their copy has run."""
    RING = 8
    _ring: list = []
    _next = 0

    @classmethod
    def send(cls, arrays, device) -> list:
        """``arrays``: numpy arrays of 4-byte elements, each [rows..]; returns device tensors of the same shapes
        and dtypes (views of one packed transfer)."""
        import numpy as np
        total = sum(a.size for a in arrays)
        if not cls._ring:
            cls._ring = [None] * cls.RING
        slot = cls._ring[cls._next]
        if slot is None or slot[0].numel() < total:
            slot = (torch.empty(max(total, 1024), dtype=torch.int32, pin_memory=True), torch.cuda.Event())
            cls._ring[cls._next] = slot
        cls._next = (cls._next + 1) % cls.RING
        host, event = slot
        event.synchronize()                       # the copy that last used this buffer has run
        flat = host.numpy()
        views, off = [], 0
        for a in arrays:
            flat[off: off + a.size] = np.ascontiguousarray(a).reshape(-1).view(np.int32)
            off += a.size
        dev = host[:total].to(device, non_blocking=True)
        event.record()
        off = 0
        for a in arrays:
            t = dev[off: off + a.size]
            views.append((t.view(torch.float32) if a.dtype == np.float32 else t).view(a.shape))
            off += a.size
        return views


def apply_penalties(logits: torch.Tensor, rows, tokens, counts, in_window, presence, frequency, repeat) -> None:
    """In place on float32 [m, vocab]: for entry i, logits[rows[i], tokens[i]] gets the presence/frequency
    penalty when counts[i] > 0 and the repetition penalty when in_window[i]; penalties are per row."""
    if _backend is not None:
        return _backend.apply_penalties(logits, rows, tokens, counts, in_window, presence, frequency, repeat)
    import numpy as np
    _dev_ok(logits)
    _need(logits.dtype == torch.float32 and logits.dim() == 2, "apply_penalties: logits must be float32 [m, vocab]")
    m, vocab = logits.shape
    n = len(rows)
    _need(len(tokens) == n and len(counts) == n and len(in_window) == n, "apply_penalties: entry lists differ in length")
    _need(len(presence) == m and len(frequency) == m and len(repeat) == m, "apply_penalties: one penalty per row")
    _need(all(0 <= r < m for r in rows), "apply_penalties: row out of range")
    dev = logits.device
    ints, fl = _Staging.send([np.asarray([rows, tokens, counts, in_window], dtype=np.int32),
                              np.asarray([presence, frequency, repeat], dtype=np.float32)], dev)
    _call("tp_apply_penalties", _ptr(logits), vocab, _ptr(ints[0]), _ptr(ints[1]), _ptr(ints[2]), _ptr(ints[3]),
          _ptr(fl[0]), _ptr(fl[1]), _ptr(fl[2]), n, _stream())


_SAMPLE_LIMITS: Optional[tuple] = None


def _sample_limits() -> tuple:
    """(pieces of a row, candidates per piece, largest top_k settled from candidates, most elements of a piece,
    bins of a counting pass) as the sampling kernels were compiled; ``sample`` sizes their scratch by these."""
    global _SAMPLE_LIMITS
    if _SAMPLE_LIMITS is None:
        buf = (ctypes.c_int * 5)()
        lib = _Library.get()
        if lib.tp_sample_limits(buf) != 0:
            raise KernelError(f"tp_sample_limits: {lib.tp_last_error().decode()}")
        _SAMPLE_LIMITS = tuple(int(v) for v in buf)
    return _SAMPLE_LIMITS


def sample(logits: torch.Tensor, work: torch.Tensor, temperature, top_k, top_p, min_p, rnd, typical_p=None,
           info: Optional[torch.Tensor] = None, settled: Optional[list] = None) -> torch.Tensor:
    """float32 [m, vocab] and per-row options (host arrays) -> int32 [m] chosen tokens.
    ``work`` is float32 scratch of at least [m, vocab].  temperature 0 rows return the argmax.
    ``typical_p`` None leaves that filter off (1.0) in every row.
    ``info``: float32 [m, 4] that receives, per row, what log-probabilities of the filtered distribution need
    (maximum, ln of the normaliser, smallest surviving value) and the chosen token's log-probability in column 3;
    ``work`` then holds the filtered, scaled logits for ``top_logprobs``.
    ``settled``: a list that receives, per row, 1 when the row was settled from the candidates of its pieces (a
    small top_k, or top_p alone on a row whose kept prefix is short) and 0 when the one block per row did it; for tests."""
    if typical_p is None:
        typical_p = [1.0] * len(temperature)
    if _backend is not None:
        if settled is not None:
            settled[:] = [0] * len(temperature)
        return _backend.sample(logits, work, temperature, top_k, top_p, min_p, rnd, typical_p, info)
    import numpy as np
    _dev_ok(logits, work)
    _need(logits.dtype == torch.float32 and logits.dim() == 2, "sample: logits must be float32 [m, vocab]")
    m, vocab = logits.shape
    _need(work.dtype == torch.float32 and work.numel() >= m * vocab, "sample: work buffer too small")
    for a in (temperature, top_k, top_p, min_p, rnd, typical_p):
        _need(len(a) == m, "sample: one option per row")
    dev = logits.device
    fl, tk = _Staging.send([np.asarray([temperature, top_p, min_p, rnd, typical_p], dtype=np.float32),
                            np.asarray(top_k, dtype=np.int32)], dev)
    out = torch.empty((m,), dtype=torch.int32, device=dev)
    # (the scratch buffers are laid out by the library's own sizes, asked of it once: pieces of a row, candidates a
    # piece may hand over, the largest top_k settled from candidates, the most elements of a piece, bins of a pass)
    pieces, ccap, kmax, per_max, bins = _sample_limits()
    part_max = torch.empty((m * pieces,), dtype=torch.float32, device=dev)    # (maxima of the pieces of each row)
    # rows that are only scaled (and cut by min_p) before the draw get the masses of their pieces from a kernel
    # of many blocks; worth it when there is such a row
    plain_rows = any(t > 0 and not (0 < k < vocab) and not (0.0 < p < 1.0) and not (ty < 1.0)
                     for t, k, p, ty in zip(temperature, top_k, top_p, typical_p))
    # rows cut by top_p alone are settled from the candidates of their pieces against the mass of the whole row
    piece_ok = -(-vocab // pieces) <= per_max and info is None
    topp_rows = piece_ok and vocab > kmax and any(
        t > 0 and not (0 < k < vocab) and 0.0 < p < 1.0 and not (ty < 1.0)
        for t, k, p, ty in zip(temperature, top_k, top_p, typical_p))
    part_mass = torch.empty((m * pieces,), dtype=torch.int64, device=dev) if (plain_rows or topp_rows) and info is None else None
    # rows cut by top_k have the first pass of their selection counted by the kernel of many blocks that scales the row
    # ... unless top_k is small: such a row is settled from the few candidates that each piece of it hands over
    small = lambda k, ty: 0 < k <= kmax and not (ty < 1.0) and piece_ok
    topk_rows = [(k, ty) for t, k, ty in zip(temperature, top_k, typical_p) if t > 0 and 0 < k < vocab]
    part_cnt = None
    if any(not small(k, ty) for k, ty in topk_rows):
        part_cnt = torch.empty((m * pieces * bins,), dtype=torch.int32, device=dev)
    cand_val = cand_idx = cand_cnt = cand_thr = done = None
    if topp_rows or any(small(k, ty) for k, ty in topk_rows):
        cand_val = torch.empty((m * pieces * ccap,), dtype=torch.float32, device=dev)
        cand_idx = torch.empty((m * pieces * ccap,), dtype=torch.int32, device=dev)
        cand_cnt = torch.empty((m * pieces,), dtype=torch.int32, device=dev)
        cand_thr = torch.empty((m * pieces,), dtype=torch.int32, device=dev)
        done = torch.empty((m,), dtype=torch.int32, device=dev)
    if info is not None:
        _dev_ok(info)
        _need(info.dtype == torch.float32 and info.is_contiguous() and tuple(info.shape) == (m, 4), "sample: info must be float32 [m, 4]")
    _call("tp_sample", _ptr(logits), _ptr(work), m, vocab, _ptr(fl[0]), _ptr(tk), _ptr(fl[1]), _ptr(fl[2]),
          _ptr(fl[4]), _ptr(fl[3]), _ptr(out), _ptr(info), _ptr(part_max), _ptr(part_mass), _ptr(part_cnt),
          _ptr(cand_val), _ptr(cand_idx), _ptr(cand_cnt), _ptr(cand_thr), _ptr(done), _stream())
    if settled is not None:
        settled[:] = [0] * m if done is None else done.tolist()
    return out


def top_logprobs(work: torch.Tensor, info: torch.Tensor, vocab: int, n: int):
    """After ``sample(..., info=info)``: the ``n`` most probable tokens of each row's filtered distribution,
    most probable first (ties by index), as (int32 [m, n] ids, float32 [m, n] log-probabilities); id -1 where a
    row has fewer survivors."""
    if _backend is not None:
        return _backend.top_logprobs(work, info, vocab, n)
    _dev_ok(work, info)
    m = info.shape[0]
    _need(info.dtype == torch.float32 and info.is_contiguous() and tuple(info.shape) == (m, 4), "top_logprobs: info must be float32 [m, 4]")
    _need(work.dtype == torch.float32 and work.is_contiguous() and work.numel() >= m * vocab, "top_logprobs: work buffer too small")
    _need(0 <= n <= vocab, "top_logprobs: n out of range")
    ids = torch.empty((m, n), dtype=torch.int32, device=info.device)
    lps = torch.empty((m, n), dtype=torch.float32, device=info.device)
    _call("tp_top_logprobs", _ptr(work), _ptr(info), m, vocab, n, _ptr(ids), _ptr(lps), _stream())
    return ids, lps


def take_rows(t: torch.Tensor, rows=None) -> torch.Tensor:
    """A new tensor holding rows ``rows`` (a list of indices; None: all of them, a plain copy) of a float32 or
    int32 tensor [n] or [n, width], by the library's own copy kernel."""
    if _backend is not None:
        return _backend.take_rows(t, rows)
    import numpy as np
    _dev_ok(t)
    _need(t.dtype in (torch.float32, torch.int32) and t.dim() in (1, 2), "take_rows: needs float32 or int32 [n] or [n, width]")
    n_in = t.shape[0]
    width = 1 if t.dim() == 1 else t.shape[1]
    if rows is None:
        n, idx = n_in, None
    else:
        n = len(rows)
        _need(all(0 <= int(r) < n_in for r in rows), "take_rows: row out of range")
        idx = _Staging.send([np.asarray(rows, dtype=np.int32)], t.device)[0] if n else None
    out = torch.empty((n,) + tuple(t.shape[1:]), dtype=t.dtype, device=t.device)
    if n and width:
        _call("tp_copy_rows4", _ptr(t), _ptr(idx), _ptr(out), n, width, _stream())
    return out


def zero_rows(t, rows) -> None:
    """t[rows] = 0 in place for a float32 or int32 tensor [n, ...], or for each of a list of them (rows: a list of indices, which
    travels to the device once)."""
    ts = [t] if isinstance(t, torch.Tensor) else list(t)
    if _backend is not None:
        for t in ts:
            _backend.zero_rows(t, rows)
        return
    import numpy as np
    _dev_ok(*ts)
    for t in ts:
        _need(t.dtype in (torch.float32, torch.int32) and t.dim() >= 1, "zero_rows: needs a float32 or int32 tensor")
        _need(all(0 <= int(r) < t.shape[0] for r in rows), "zero_rows: row out of range")
    idx = None
    for t in ts:
        width = t[0].numel() if t.shape[0] else 0
        if len(rows) and width:
            if idx is None or idx.device != t.device:
                idx = _Staging.send([np.asarray(rows, dtype=np.int32)], t.device)[0]
            _call("tp_zero_rows4", _ptr(t), _ptr(idx), len(rows), width, _stream())


def fill_normal(out: torch.Tensor, seed: int, mean: float, std: float) -> torch.Tensor:
    """Fill a device tensor with mean + std * N(0, 1); element i depends only on (seed, i) and has the bits
    that ``weights.random_init.fill_normal_host`` gives it on the host."""
    if _backend is not None:
        return _backend.fill_normal(out, seed, mean, std)
    _dev_ok(out)
    _call("tp_fill_normal", _ptr(out), _dt(out), int(out.numel()), ctypes.c_ulonglong(seed & (2 ** 64 - 1)),
          ctypes.c_double(mean), ctypes.c_double(std), _stream())
    return out


# ---------------------------------------------------------------------------------
# Operations of layers with a hashed bigram embedding, norms behind the sublayers, a gated delta-rule mixer and
# routed experts.

def embed_bigram(tokens: torch.Tensor, table: torch.Tensor, bigram: Optional[torch.Tensor], positions: torch.Tensor,
                 token_req: torch.Tensor, cu_seqlens: torch.Tensor, state_slots: torch.Tensor, prev_state: torch.Tensor,
                 num_requests: int, mul_prev: int, mul_cur: int, buckets: int, scale: float = 1.0,
                 pos_table: Optional[torch.Tensor] = None) -> torch.Tensor:
    """float32 [n, hidden] = table[token] * scale + bigram[row], row = (previous * mul_prev + token * mul_cur) mod buckets,
    and row ``buckets`` for a token at position 0.  The previous token of a run's first token is what
    ``prev_state`` (int32 [slots, 1]) holds for the request's slot; each run's last token is left there.
    ``pos_table`` ([positions, hidden], of the tables' type): its row of the token's position is added as well.
    ``bigram`` None: no second row (and nothing is read from or left in ``prev_state``, which may be None too)."""
    if _backend is not None:
        if scale != 1.0 or pos_table is not None:
            return _backend.embed_bigram(tokens, table, bigram, positions, token_req, cu_seqlens, state_slots, prev_state,
                                         num_requests, mul_prev, mul_cur, buckets, scale, pos_table)
        return _backend.embed_bigram(tokens, table, bigram, positions, token_req, cu_seqlens, state_slots, prev_state,
                                     num_requests, mul_prev, mul_cur, buckets)
    _dev_ok(tokens, table, bigram, positions, token_req, cu_seqlens, state_slots, prev_state, pos_table)
    n = tokens.numel()
    _need(pos_table is None or (pos_table.dim() == 2 and pos_table.shape[1] == table.shape[1] and pos_table.dtype == table.dtype),
          "embed_bigram: the position table must be [positions, hidden] of the tables' type")
    _need(table.dim() == 2, "embed_bigram: tables must be [rows, hidden] of one type")
    if bigram is not None:
        _need(bigram.dim() == 2 and bigram.shape[1] == table.shape[1] and bigram.dtype == table.dtype,
              "embed_bigram: tables must be [rows, hidden] of one type")
        if not (bigram.shape[0] == buckets + 1):
            raise KernelError(f"embed_bigram: the bigram table needs {buckets + 1} rows, has {bigram.shape[0]}")
        _need(prev_state is not None and prev_state.dtype == torch.int32, "embed_bigram: the state must be int32")
    _i32(tokens, n, "embed tokens") if n else None
    _i32(positions, n, "embed positions") if n else None
    _i32(token_req, n, "token_req") if n else None
    _i32(cu_seqlens, num_requests + 1, "cu_seqlens")
    _i32(state_slots, num_requests, "state_slots")
    hidden = table.shape[1]
    out = torch.empty((n, hidden), dtype=torch.float32, device=table.device)
    _call("tp_embed_bigram", _ptr(tokens), _ptr(positions), _ptr(token_req), _ptr(cu_seqlens), _ptr(state_slots), _ptr(prev_state),
          _ptr(table), _ptr(bigram), _dt(table), _ptr(out), n, int(num_requests), hidden, ctypes.c_longlong(mul_prev),
          ctypes.c_longlong(mul_cur), ctypes.c_longlong(buckets), float(scale), _ptr(pos_table), _stream())
    return out


def sigmoid_gate(a: torch.Tensor, proj: Optional[torch.Tensor], gate_col0: int, scale: float, out: torch.Tensor, out_col0: int,
                 per: int = 1) -> None:
    """out[:, out_col0 + c] = a[:, c] * sigmoid(proj[:, gate_col0 + c // per]) * scale (``proj`` float32 rows; None: no
    gate; ``per`` columns in a row share a gate); ``a`` and ``out`` are of one type, ``out`` [n, wider]."""
    if _backend is not None:
        if per != 1:
            return _backend.sigmoid_gate(a, proj, gate_col0, scale, out, out_col0, per)
        return _backend.sigmoid_gate(a, proj, gate_col0, scale, out, out_col0)
    _dev_ok(a, proj, out)
    _need(a.dim() == 2 and out.dim() == 2 and a.dtype == out.dtype and a.shape[0] == out.shape[0], "sigmoid_gate: bad operands")
    n, width = a.shape
    _need(0 <= out_col0 and out_col0 + width <= out.shape[1], "sigmoid_gate: output rows too short")
    _need(per >= 1 and width % per == 0, "sigmoid_gate: columns are no whole runs of per")
    if proj is not None:
        _need(proj.dtype == torch.float32 and proj.dim() == 2 and proj.shape[0] == n and 0 <= gate_col0 and gate_col0 + width // per <= proj.shape[1],
              "sigmoid_gate: bad gate rows")
    _call("tp_sigmoid_gate", _ptr(a), _dt(a), _ptr(proj), 0 if proj is None else proj.shape[1], int(gate_col0), float(scale),
          _ptr(out), out.shape[1], int(out_col0), n, width, int(per), _stream())


def turn_gate(a: torch.Tensor, positions: torch.Tensor, inv_freq: torch.Tensor, dim: int, gate: Optional[torch.Tensor] = None,
              gate_col0: int = 0, cos_sin: Optional[torch.Tensor] = None) -> torch.Tensor:
    """a [n, heads * dim] with every head's pairs of neighbours (2 m, 2 m + 1) turned by -positions * inv_freq[m], times
    sigmoid(gate[:, gate_col0 + c]) when ``gate`` (float32 rows) is given; same type.  ``inv_freq`` float64 [dim / 2];
    ``cos_sin``: this step's table of its angles (``rope_table``)."""
    if _backend is not None:
        return _backend.turn_gate(a, positions, inv_freq, dim, gate, gate_col0)
    _dev_ok(a, positions, inv_freq, gate, cos_sin)
    _need(a.dim() == 2 and dim > 0 and dim % 2 == 0 and a.shape[1] % dim == 0, "turn_gate: rows must be whole heads of an even size")
    n, width = a.shape
    _i32(positions, n, "positions") if n else None
    _need(inv_freq.dtype == torch.float64 and inv_freq.numel() == dim // 2, "turn_gate: inv_freq must be float64 [dim / 2]")
    if gate is not None:
        _need(gate.dtype == torch.float32 and gate.dim() == 2 and gate.shape[0] == n and 0 <= gate_col0 and gate_col0 + width <= gate.shape[1],
              "turn_gate: bad gate rows")
    if cos_sin is not None:
        _need(cos_sin.dtype == torch.float32 and tuple(cos_sin.shape) == (n, dim // 2, 2), "turn_gate: table must be float32 [n, dim / 2, 2]")
    out = torch.empty_like(a)
    _call("tp_turn_gate", _ptr(a), _dt(a), _ptr(positions), _ptr(inv_freq), _ptr(cos_sin), _ptr(gate),
          int(0 if gate is None else gate.shape[1]), int(gate_col0), _ptr(out), n, width // dim, int(dim), _stream())
    return out


def _cache_pair(k_cache, v_cache, kv_heads, key_dim, value_dim, what):
    if not (k_cache.dim() == 4 and v_cache.dim() == 4 and k_cache.shape[1] == kv_heads and k_cache.shape[3] == key_dim
            and tuple(v_cache.shape) == (k_cache.shape[0], kv_heads, value_dim, k_cache.shape[2]) and v_cache.dtype == k_cache.dtype):
        raise KernelError(f"{what}: caches must be k [pages, {kv_heads}, page_size, {key_dim}], v [pages, {kv_heads}, {value_dim}, page_size] of one type")


def _rotation(inv_freq, pairs, cos_sin, n, what):
    if pairs:
        if not (inv_freq is not None and inv_freq.dtype == torch.float64 and inv_freq.numel() == pairs):
            raise KernelError(f"{what}: frequencies must be float64 [{pairs}]")
    if cos_sin is not None:
        if not (cos_sin.dtype == torch.float32 and tuple(cos_sin.shape) == (n, pairs, 2)):
            raise KernelError(f"{what}: table must be float32 [n, {pairs}, 2]")


def qkv_rows(rows: torch.Tensor, positions: torch.Tensor, slots: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int,
             value_dim: int, k_cache: torch.Tensor, v_cache: torch.Tensor, inv_freq: Optional[torch.Tensor] = None, rotary_dim: int = 0,
             factor: float = 1.0, cos_sin: Optional[torch.Tensor] = None, biases=(None, None, None), norms=None, eps: float = 0.0,
             value_inv_freq: Optional[torch.Tensor] = None, value_cos_sin: Optional[torch.Tensor] = None,
             pad_dim: Optional[int] = None, col0: int = 0, norm_over: str = "projection") -> torch.Tensor:
    """Float32 rows [n, q | k | v | any more columns] of a projection, step by step: ``biases`` (float32 per column of q, k,
    v; each may be None) are added; with ``norms`` (q weight, k weight: float32, one value a column) q and k are divided
    by the root mean square of the WHOLE projection (all heads together, ``eps`` inside the root) and multiplied by the
    weight (``norm_over`` ``"head"``: every head by its own root mean square, the weights [head_dim] shared by the heads); the
    pairs of neighbours of the first ``rotary_dim`` elements of q and k heads turn by position *
    ``inv_freq``; with ``value_inv_freq`` (float64 [value_dim / 2]) the pairs of a value head turn likewise; k and v go
    to the cache rows ``slots``.  Returns q in the caches' type as [n, heads, pad_dim or head_dim] (keys are stored as
    wide; zeros behind a head's own elements).  ``col0``: the column at which q | k | v start."""
    od = head_dim if pad_dim is None else int(pad_dim)
    if not (norm_over in ("projection", "head")):
        raise KernelError(f"qkv_rows: norm over {norm_over!r} unknown")
    per_head = norm_over == "head"
    if _backend is not None:
        if col0 or per_head:
            return _backend.qkv_rows(rows, positions, slots, num_heads, num_kv_heads, head_dim, value_dim, k_cache, v_cache, inv_freq,
                                     rotary_dim, factor, biases, norms, eps, value_inv_freq, od, col0, norm_over)
        return _backend.qkv_rows(rows, positions, slots, num_heads, num_kv_heads, head_dim, value_dim, k_cache, v_cache, inv_freq,
                                 rotary_dim, factor, biases, norms, eps, value_inv_freq, od)
    qb, kb, vb = biases
    qn, kn = norms if norms is not None else (None, None)
    _dev_ok(rows, positions, slots, k_cache, v_cache, inv_freq, cos_sin, qb, kb, vb, qn, kn, value_inv_freq, value_cos_sin)
    n = rows.shape[0]
    widths = (num_heads * head_dim, num_kv_heads * head_dim, num_kv_heads * value_dim)
    _need(rows.dtype == torch.float32 and rows.dim() == 2 and col0 >= 0 and rows.shape[1] >= col0 + sum(widths) and rows.shape[1] % 2 == 0,
          "qkv_rows: rows must be float32 [n, an even width of at least q | k | v]")
    for b, size, what in ((qb, widths[0], "q bias"), (kb, widths[1], "k bias"), (vb, widths[2], "v bias"),
                          (qn, head_dim if per_head else widths[0], "q norm"), (kn, head_dim if per_head else widths[1], "k norm")):
        if not (b is None or (b.dtype == torch.float32 and b.numel() == size)):
            raise KernelError(f"qkv_rows: {what} must be float32 with {size} elements")
    _need((qn is None) == (kn is None), "qkv_rows: the norms of q and k come together")
    if n:
        _i32(positions, n, "positions")
        _i32(slots, n, "slots")
    _need(head_dim % 2 == 0 and value_dim % 2 == 0 and od >= head_dim and od % 2 == 0, "qkv_rows: head sizes must be even")
    _need(0 <= rotary_dim <= head_dim and rotary_dim % 2 == 0, "qkv_rows: bad rotary_dim")
    _cache_pair(k_cache, v_cache, num_kv_heads, od, value_dim, "qkv_rows")
    _rotation(inv_freq, rotary_dim // 2, cos_sin, n, "qkv_rows")
    if value_inv_freq is not None:
        _rotation(value_inv_freq, value_dim // 2, value_cos_sin, n, "qkv_rows: values")
    q = torch.empty((n, num_heads, od), dtype=k_cache.dtype, device=rows.device)
    _call("tp_qkv_rows", (rows.data_ptr() + 4 * int(col0)), int(rows.shape[1]), int(rows.shape[1] - int(col0)),
          _ptr(qb), _ptr(kb), _ptr(vb), _ptr(qn), _ptr(kn), float(eps),
          _ptr(positions), _ptr(slots), _ptr(inv_freq), _ptr(cos_sin), int(rotary_dim), float(factor), _ptr(value_inv_freq),
          _ptr(value_cos_sin), n, int(num_heads), int(num_kv_heads), int(head_dim), int(value_dim), od, _ptr(q), _ptr(k_cache),
          _ptr(v_cache), _dt(k_cache), k_cache.shape[2], int(per_head), _stream())
    return q


def latent_rows_write(rows: torch.Tensor, q_col0: int, d_col0: int, weight: torch.Tensor, eps: float, positions: torch.Tensor,
                      slots: torch.Tensor, inv_freq: Optional[torch.Tensor], factor: float, num_heads: int, rotary_dim: int,
                      latent_dim: int, k_cache: torch.Tensor, v_cache: torch.Tensor,
                      cos_sin: Optional[torch.Tensor] = None, plain_dim: Optional[int] = None) -> torch.Tensor:
    """Float32 rows [n, width]: queries at ``q_col0``, per head [rotary_dim | latent_dim] elements (``plain_dim`` given: per
    head [plain_dim | rotary_dim] elements of which only the rotary ones are taken; the latent part of the result is left
    for the caller to fill), and at ``d_col0`` a latent before its norm [latent_dim] followed by one shared rotated key part [rotary_dim].  The latent is RMS-normed
    (``weight``, ``eps``), the rotary elements of the queries and of the key part turn (pairs of neighbours, position *
    ``inv_freq``); the cache rows ``slots`` get keys [rotated | latent | zeros] (one head) and, transposed, values
    [latent | zeros]; the sizes of both are the caches' own.  Returns q [n, heads, key size], laid out like the keys."""
    if _backend is not None:
        return _backend.latent_rows_write(rows, q_col0, d_col0, weight, eps, positions, slots, inv_freq, factor, num_heads, rotary_dim,
                                          latent_dim, k_cache, v_cache, plain_dim)
    _dev_ok(rows, weight, positions, slots, inv_freq, k_cache, v_cache, cos_sin)
    n, key = rows.shape[0], rotary_dim + latent_dim
    q_head, q_rot = (key, 0) if plain_dim is None else (int(plain_dim) + rotary_dim, int(plain_dim))
    _need(rows.dtype == torch.float32 and rows.dim() == 2 and rows.shape[1] % 2 == 0 and q_col0 >= 0 and q_col0 % 2 == 0 and d_col0 >= 0
          and q_head % 2 == 0 and q_rot % 2 == 0 and q_col0 + num_heads * q_head <= rows.shape[1] and d_col0 + key <= rows.shape[1], "latent_rows_write: bad rows")
    _need(weight.dtype == torch.float32 and weight.numel() == latent_dim, "latent_rows_write: weight must be float32 [latent_dim]")
    _need(k_cache.dim() == 4 and v_cache.dim() == 4, "latent_rows_write: bad caches")
    od, vd = k_cache.shape[3], v_cache.shape[2]
    _need(rotary_dim % 2 == 0 and key % 2 == 0 and od >= key and od % 2 == 0 and vd >= latent_dim, "latent_rows_write: bad head sizes")
    _cache_pair(k_cache, v_cache, 1, od, vd, "latent_rows_write")
    _rotation(inv_freq, rotary_dim // 2, cos_sin, n, "latent_rows_write")
    if n:
        _i32(positions, n, "positions")
        _i32(slots, n, "slots")
    q = torch.empty((n, num_heads, od), dtype=k_cache.dtype, device=rows.device)
    _call("tp_latent_rows_write", _ptr(rows), int(rows.shape[1]), int(q_col0), int(d_col0), _ptr(weight), float(eps),
          _ptr(positions), _ptr(slots), _ptr(inv_freq), _ptr(cos_sin), float(factor), n, int(num_heads), int(rotary_dim),
          int(latent_dim), od, vd, _ptr(q), _ptr(k_cache), _ptr(v_cache), _dt(k_cache), k_cache.shape[2], q_head, q_rot,
          int(plain_dim is None), _stream())
    return q


def head_linear_ok(n: int, k: int, dtype: torch.dtype) -> bool:
    """Whether ``head_linear`` takes weights [heads, n, k]."""
    return allow_mfma and dtype == torch.bfloat16 and k % 32 == 0 and n % 16 == 0


def head_linear(x: torch.Tensor, x_col0: int, x_head: int, w: torch.Tensor, out: torch.Tensor, out_col0: int, out_head: int,
                gate: Optional[torch.Tensor] = None, gate_col0: int = 0, scale: float = 1.0) -> None:
    """A product per head: out[m, out_col0 + h * out_head + n] = scale * sigmoid(gate[m, gate_col0 + h]) * sum_k w[h, n, k] *
    x[m, x_col0 + h * x_head + k], for bfloat16 weights [heads, n, k], rows ``x`` (float32 or bfloat16; float32 is rounded to
    bfloat16) and bfloat16 rows ``out``; ``gate`` float32 rows or None.  Sizes: ``head_linear_ok``."""
    if _backend is not None:
        return _backend.head_linear(x, x_col0, x_head, w, out, out_col0, out_head, gate, gate_col0, scale)
    _dev_ok(x, w, out, gate)
    _need(w.dim() == 3 and w.dtype == torch.bfloat16 and head_linear_ok(w.shape[1], w.shape[2], w.dtype), "head_linear: bad weights")
    H, N, K = w.shape
    _need(x.dim() == 2 and out.dim() == 2 and out.dtype == torch.bfloat16 and x.shape[0] == out.shape[0], "head_linear: bad rows")
    _need(0 <= x_col0 and x_col0 + (H - 1) * x_head + K <= x.shape[1] and x_head >= K, "head_linear: input rows too short")
    _need(0 <= out_col0 and out_col0 + (H - 1) * out_head + N <= out.shape[1] and out_head >= N, "head_linear: output rows too short")
    m = x.shape[0]
    if gate is not None:
        _need(gate.dtype == torch.float32 and gate.dim() == 2 and gate.shape[0] == m and 0 <= gate_col0 and gate_col0 + H <= gate.shape[1],
              "head_linear: bad gate rows")
    at = lambda t, col: (t.data_ptr() + col * t.element_size())
    _call("tp_head_linear", at(x, x_col0), _dt(x), int(x.shape[1]), int(x_head), _ptr(w), at(out, out_col0),
          int(out.shape[1]), int(out_head), _ptr(None) if gate is None else at(gate, gate_col0),
          int(0 if gate is None else gate.shape[1]), float(scale), m, H, N, K, _stream(), tag=(m, H, N, K))


def norm_add(h: torch.Tensor, y: torch.Tensor, weight: torch.Tensor, eps: float, next_weight: Optional[torch.Tensor] = None,
             next_eps: float = 0.0, out_dtype: Optional[torch.dtype] = None, gate: Optional[torch.Tensor] = None, gate_col0: int = 0,
             gate_bias: Optional[torch.Tensor] = None, normed: bool = True, blocked: bool = False):
    """h += y / sqrt(mean(y^2) + eps) * weight (not ``normed``: h += y * weight), per row, in place (float32 [n, width]; y may be
    ``Partials``).  With ``next_weight`` the
    rows of the new h normed with it (and ``next_eps``) come back as ``out_dtype``.  With ``gate`` (float32 rows [n,
    wider]) y is first multiplied by sigmoid(gate[:, gate_col0 + c] + gate_bias[c]).  ``blocked``: the rows come back as
    ``KBlocked`` (see ``few_rows_ok``)."""
    if _backend is not None:
        if gate is not None:
            return _backend.norm_add(h, y, weight, eps, next_weight, next_eps, out_dtype, gate, gate_col0, gate_bias)
        return _backend.norm_add(h, y, weight, eps, next_weight, next_eps, out_dtype)
    parts = 1
    if isinstance(y, Partials):
        parts, y = y.data.shape[0], y.data.view(-1, y.data.shape[2])
        _need(y.shape[0] == parts * h.shape[0] and y.is_contiguous(), "norm_add: malformed partial sums")
    _dev_ok(h, y, weight, next_weight, gate, gate_bias)
    _need(h.dtype == torch.float32 and h.dim() == 2 and y.dtype == torch.float32 and tuple(y.shape) == (parts * h.shape[0], h.shape[1]),
          "norm_add: h and y must be float32 [n, width]")
    n, width = h.shape
    _need(weight.dtype == torch.float32 and weight.numel() == width, "norm_add: weight must be float32 [width]")
    if gate is not None:
        _need(gate.dtype == torch.float32 and gate.dim() == 2 and gate.shape[0] == n and 0 <= gate_col0 and gate_col0 + width <= gate.shape[1],
              "norm_add: bad gate rows")
        _need(gate_bias is None or (gate_bias.dtype == torch.float32 and gate_bias.numel() == width), "norm_add: gate bias must be float32 [width]")
    x = None
    if next_weight is not None:
        _need(next_weight.dtype == torch.float32 and next_weight.numel() == width and out_dtype is not None, "norm_add: bad next norm")
        x = torch.empty((width // 8, n, 8) if blocked else (n, width), dtype=out_dtype, device=h.device)
    _call("tp_norm_add", _ptr(h), _ptr(y), _ptr(weight), float(eps), _ptr(next_weight), float(next_eps), _ptr(x),
          _dtcode(out_dtype) if x is not None else _F32, n, width, _ptr(gate), int(0 if gate is None else gate.shape[1]),
          int(gate_col0), _ptr(gate_bias), int(normed), int(blocked), parts, _stream())
    return KBlocked(x, n, width) if blocked and x is not None else x


def scale_add(h: torch.Tensor, y: torch.Tensor, weight: torch.Tensor, next_weight: Optional[torch.Tensor] = None, next_eps: float = 0.0,
              out_dtype: Optional[torch.dtype] = None, gate: Optional[torch.Tensor] = None, gate_col0: int = 0,
              gate_bias: Optional[torch.Tensor] = None, blocked: bool = False):
    """``norm_add`` without the norm on y: h += y * weight, per row, in place (``weight`` a vector of scales), and with
    ``next_weight`` the rows of the new h normed with it come back."""
    if _backend is not None:
        return _backend.scale_add(h, y, weight, next_weight, next_eps, out_dtype, gate, gate_col0, gate_bias)
    return norm_add(h, y, weight, 0.0, next_weight, next_eps, out_dtype, gate, gate_col0, gate_bias, normed=False, blocked=blocked)


ACTIVATIONS = {"gelu_tanh": 0, "silu": 1, "gelu_erf": 2, "relu2": 3}


def activation(u: torch.Tensor, kind: str, out_dtype: torch.dtype, col0: int = 0, width: Optional[int] = None,
               gate_col: Optional[int] = None, blocked: bool = False):
    """Element by element: ``gelu_tanh`` (0.5 z (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3)))), ``gelu_erf``
    (0.5 z (1 + erf(z / sqrt(2)))), ``relu2`` (max(z, 0)^2) or ``silu``, formed in float32, as ``out_dtype``.
    With ``width`` (``u`` float32 rows [n, wider]): the columns col0 .. col0 + width of every row, and with ``gate_col``
    each row's results times the sigmoid of that column of the row.  ``blocked`` (whole float32 rows, see ``few_rows_ok``):
    the result comes as ``KBlocked``."""
    if not (kind in ACTIVATIONS):
        raise KernelError(f"activation: {kind!r} unknown (known: {sorted(ACTIVATIONS)})")
    if _backend is not None:
        if width is not None:
            return _backend.activation(u, kind, out_dtype, col0, width, gate_col)
        return _backend.activation(u, kind, out_dtype)
    _dev_ok(u)
    if width is not None:
        _need(u.dtype == torch.float32 and u.dim() == 2 and 0 <= col0 and col0 + width <= u.shape[1] and width > 0,
              "activation: rows must be float32 [n, wider]")
        _need(gate_col is None or 0 <= gate_col < u.shape[1], "activation: gate column outside the rows")
        out = torch.empty((u.shape[0], width), dtype=out_dtype, device=u.device)
        _call("tp_activation_rows", _ptr(u), int(u.shape[1]), int(col0), int(width), -1 if gate_col is None else int(gate_col),
              _ptr(out), _dtcode(out_dtype), u.shape[0], ACTIVATIONS[kind], _stream())
        return out
    if blocked:
        _need(u.dim() == 2 and u.dtype == torch.float32 and u.shape[1] % 8 == 0, "activation: k-blocked results need whole float32 rows")
        m, n = u.shape
        out = torch.empty((n // 8, m, 8), dtype=out_dtype, device=u.device)
        _call("tp_activation_blocked", _ptr(u), _ptr(out), _dtcode(out_dtype), m, n, ACTIVATIONS[kind], _stream())
        return KBlocked(out, m, n)
    out = torch.empty(u.shape, dtype=out_dtype, device=u.device)
    _call("tp_activation", _ptr(u), _dt(u), _ptr(out), _dtcode(out_dtype), int(u.numel()), ACTIVATIONS[kind], _stream())
    return out


ROUTE_SCORES = {"softmax": 0, "sigmoid": 1}


def moe_route(logits: torch.Tensor, correction: Optional[torch.Tensor], experts: int, top: int, groups: int, keep: int,
              score: str = "softmax", group_best: int = 1, normalize: bool = False, sum_eps: float = 0.0, scale: float = 1.0,
              bias: Optional[torch.Tensor] = None):
    """Router of a mixture of experts over float32 logits [n, >= experts]: s = softmax over the experts (``score``
    ``"sigmoid"``: the sigmoid of each logit by itself); an expert's choice score is s + correction (None: s); with
    ``groups`` > 1 only the experts of the ``keep`` groups (of neighbours) whose ``group_best`` largest choice scores
    add up highest can be chosen; the ``top`` best allowed experts are chosen and weigh s, with ``normalize`` divided by
    the chosen experts' sum (+ ``sum_eps``), times ``scale``.  Returns (dense float32 [n, experts] with a chosen expert's
    weight and 0 elsewhere, ids int32 [n, top], weights [n, top]).  ``bias`` (float32 [experts]) is added to the logits
    first.  (A softmax over the chosen logits alone is ``normalize`` without ``sum_eps``: the chosen experts' shares of
    the full softmax over their sum.)"""
    if not (score in ROUTE_SCORES):
        raise KernelError(f"moe_route: score {score!r} unknown")
    if _backend is not None:
        if bias is not None:
            return _backend.moe_route(logits, correction, experts, top, groups, keep, score, group_best, normalize, sum_eps, scale, bias)
        if (score, group_best, normalize, scale) == ("softmax", 1, False, 1.0) and correction is not None:
            return _backend.moe_route(logits, correction, experts, top, groups, keep)
        return _backend.moe_route(logits, correction, experts, top, groups, keep, score, group_best, normalize, sum_eps, scale)
    _dev_ok(logits, correction, bias)
    _need(bias is None or (bias.dtype == torch.float32 and bias.numel() == experts), "moe_route: bias must be float32 [experts]")
    _need(logits.dtype == torch.float32 and logits.dim() == 2 and logits.shape[1] >= experts, "moe_route: logits must be float32 [n, experts]")
    _need(correction is None or (correction.dtype == torch.float32 and correction.numel() == experts), "moe_route: correction must be float32 [experts]")
    _need(group_best >= 1, "moe_route: group_best must be at least 1")
    n = logits.shape[0]
    dense = torch.empty((n, experts), dtype=torch.float32, device=logits.device)
    ids = torch.empty((n, top), dtype=torch.int32, device=logits.device)
    weights = torch.empty((n, top), dtype=torch.float32, device=logits.device)
    _call("tp_moe_route", _ptr(logits), logits.shape[1], _ptr(correction), int(experts), int(top), int(groups), int(keep), _ptr(dense),
          _ptr(ids), _ptr(weights), n, ROUTE_SCORES[score], int(group_best), int(bool(normalize)), float(sum_eps),
          float(scale), _ptr(bias), _stream())
    return dense, ids, weights


LOWRANK_MODES = {"plain": 0, "sigmoid": 1, "decay": 2, "rate_sigmoid": 3, "exp_exp": 4, "root_sigmoid": 5}


def lowrank_up(x: torch.Tensor, col0: int, weight_t: torch.Tensor, mode: str = "plain", a_log: Optional[torch.Tensor] = None,
               bias: Optional[torch.Tensor] = None, per_head: int = 0, rate: float = 0.0, in_act: Optional[str] = None) -> torch.Tensor:
    """The second product of a low-rank projection: float32 [n, N] = f(g(x[:, col0: col0 + r]) @ weight_t), ``x`` float32
    rows (the first product's sums), ``weight_t`` float32 [r, N].  f: ``plain``; ``sigmoid``; ``decay``:
    exp(-exp(a_log[c // per_head]) * softplus(sum + bias[c])); ``rate_sigmoid``: exp(-rate * sigmoid(sum + bias[c]));
    ``exp_exp``: exp(-exp(sum + bias[c])); ``root_sigmoid``: sigmoid(sum + bias[c])^rate.
    g: the identity, or tanh with ``in_act`` ``"tanh"``."""
    if not (in_act in (None, "tanh")):
        raise KernelError(f"lowrank_up: input function {in_act!r} unknown")
    if _backend is not None:
        if mode in ("rate_sigmoid", "exp_exp", "root_sigmoid") or in_act is not None:
            return _backend.lowrank_up(x, col0, weight_t, mode, a_log, bias, per_head, rate, in_act)
        return _backend.lowrank_up(x, col0, weight_t, mode, a_log, bias, per_head)
    _dev_ok(x, weight_t, a_log, bias)
    if not (mode in LOWRANK_MODES):
        raise KernelError(f"lowrank_up: mode {mode!r} unknown")
    _need(x.dtype == torch.float32 and x.dim() == 2 and weight_t.dtype == torch.float32 and weight_t.dim() == 2, "lowrank_up: float32 operands")
    r, n_out = weight_t.shape
    _need(0 <= col0 and col0 + r <= x.shape[1], "lowrank_up: rows too short")
    if mode == "decay":
        _need(a_log is not None and bias is not None and per_head > 0 and n_out % per_head == 0 and a_log.dtype == torch.float32
              and bias.dtype == torch.float32 and a_log.numel() == n_out // per_head and bias.numel() == n_out, "lowrank_up: bad decay constants")
    if mode in ("rate_sigmoid", "exp_exp", "root_sigmoid"):
        _need(bias is not None and bias.dtype == torch.float32 and bias.numel() == n_out, "lowrank_up: bad decay biases")
    out = torch.empty((x.shape[0], n_out), dtype=torch.float32, device=x.device)
    _call("tp_lowrank_up", _ptr(x), x.shape[1], int(col0), r, _ptr(weight_t), _ptr(out), x.shape[0], n_out, LOWRANK_MODES[mode],
          _ptr(a_log), _ptr(bias), int(per_head), 1 if in_act == "tanh" else 0, float(rate), _stream())
    return out


def delta_scan(qkv: torch.Tensor, decay: torch.Tensor, proj: torch.Tensor, beta_col0: int, state: torch.Tensor, state_off: int,
               cu_seqlens: torch.Tensor, state_slots: torch.Tensor, num_requests: int, heads: int, kv_heads: int, dim: int,
               vdim: int, q_scale: float, unit_eps: float, max_run: int = 0) -> torch.Tensor:
    """The gated delta rule per head over each request's run.  ``qkv`` float32 [n, q | k | v] with q and k
    [kv_heads * dim] and v [heads * vdim]; q and k are made unit vectors per head (x / sqrt(sum x^2 + unit_eps), q times
    ``q_scale``); beta = sigmoid(proj[:, beta_col0 + h]); ``decay`` float32 [n, heads * dim].  Per head, with S
    [dim, vdim] (kept at ``state[slot, state_off:]`` column by column, [heads, vdim, dim]):  S <- decay * S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q.
    Returns o float32 [n, heads * vdim]; the state is left as the run leaves it.  (q and k of ``qkv`` may be left as
    unit vectors: the rows are a temporary of the caller's.)  ``max_run``: the longest run (0: not known); runs of 64
    tokens and more go by groups of tokens, which changes rounding only, whatever runs stand beside them."""
    if _backend is not None:
        return _backend.delta_scan(qkv, decay, proj, beta_col0, state, state_off, cu_seqlens, state_slots, num_requests, heads,
                                   kv_heads, dim, vdim, q_scale, unit_eps)
    _dev_ok(qkv, decay, proj, state, cu_seqlens, state_slots)
    n = qkv.shape[0]
    _need(qkv.dtype == torch.float32 and qkv.dim() == 2 and qkv.shape[1] == 2 * kv_heads * dim + heads * vdim, "delta_scan: bad q | k | v rows")
    _need(decay.dtype == torch.float32 and tuple(decay.shape) == (n, heads * dim), "delta_scan: decay must be float32 [n, heads * dim]")
    _need(proj.dtype == torch.float32 and proj.dim() == 2 and proj.shape[0] == n and 0 <= beta_col0 and beta_col0 + heads <= proj.shape[1],
          "delta_scan: bad projection rows")
    _need(state.dtype == torch.float32 and state.dim() == 2 and state_off >= 0 and state.shape[1] >= state_off + heads * dim * vdim,
          "delta_scan: state rows too short")
    _i32(cu_seqlens, num_requests + 1, "cu_seqlens")
    _i32(state_slots, num_requests, "state_slots")
    y = torch.empty((n, heads * vdim), dtype=torch.float32, device=qkv.device)
    kq = torch.empty((n, kv_heads), dtype=torch.float32, device=qkv.device)      # k . q per token and key head
    max_run = min(int(max_run), n)
    need = library().tp_delta_scan_scratch(n, int(num_requests), max_run, int(heads), int(dim), int(vdim)) if allow_mfma else 0
    scratch = torch.empty((need,), dtype=torch.float32, device=qkv.device) if need else None
    _call("tp_delta_scan", _ptr(qkv), qkv.shape[1], _ptr(decay), _ptr(proj), proj.shape[1], int(beta_col0), _ptr(state),
          int(state.shape[1]), int(state_off), _ptr(cu_seqlens), _ptr(state_slots), _ptr(y), _ptr(kq), n,
          int(num_requests), int(heads), int(kv_heads), int(dim), int(vdim), float(q_scale), float(unit_eps),
          max_run, _ptr(scratch), int(need), _stream())
    return y


GATE_ACTS = {"sigmoid": 1, "silu": 2}


def head_norm_gate(o: torch.Tensor, weight: torch.Tensor, gate: Optional[torch.Tensor], eps: float, scale: float, heads: int,
                   out: torch.Tensor, out_col0: int, gate_rows: Optional[torch.Tensor] = None, gate_col0: int = 0,
                   gate_act: str = "sigmoid") -> None:
    """out[:, out_col0 + h * vdim + d] = o[:, h, d] / sqrt(mean_d o^2 + eps) * weight[d] * gate[:, h * vdim + d] * scale:
    ``o`` float32 [n, heads * vdim]; ``weight`` float32 [vdim] shared by the heads, or [heads * vdim], every head its own;
    ``gate`` float32 like ``o`` or None.  ``gate_rows`` (float32 rows [n, wider], instead of ``gate``): the gate is the
    sigmoid (``gate_act`` ``"silu"``: the SiLU) of their columns gate_col0 .. gate_col0 + heads * vdim."""
    if not (gate_act in GATE_ACTS):
        raise KernelError(f"head_norm_gate: gate function {gate_act!r} unknown (known: {sorted(GATE_ACTS)})")
    if _backend is not None:
        if gate_act != "sigmoid":
            return _backend.head_norm_gate(o, weight, gate, eps, scale, heads, out, out_col0, gate_rows, gate_col0, gate_act)
        if gate_rows is not None:
            return _backend.head_norm_gate(o, weight, gate, eps, scale, heads, out, out_col0, gate_rows, gate_col0)
        return _backend.head_norm_gate(o, weight, gate, eps, scale, heads, out, out_col0)
    _dev_ok(o, weight, gate, out, gate_rows)
    _need(o.dtype == torch.float32 and o.dim() == 2 and o.shape[1] % heads == 0, "head_norm_gate: o must be float32 [n, heads * vdim]")
    n, vdim = o.shape[0], o.shape[1] // heads
    _need(weight.dtype == torch.float32 and weight.numel() in (vdim, heads * vdim), "head_norm_gate: weight must be float32 [vdim] or [heads * vdim]")
    # (one head: a weight of [vdim] is both)
    per_head = int(weight.numel() == heads * vdim and heads > 1)
    _need(gate is None or gate_rows is None, "head_norm_gate: one gate")
    _need(gate is None or (gate.dtype == torch.float32 and tuple(gate.shape) == tuple(o.shape)), "head_norm_gate: gate must match o")
    _need(out.dim() == 2 and out.shape[0] == n and 0 <= out_col0 and out_col0 + o.shape[1] <= out.shape[1], "head_norm_gate: output rows too short")
    gate_ptr, gate_stride, raw = _ptr(gate), o.shape[1], 0
    if gate_rows is not None:
        _need(gate_rows.dtype == torch.float32 and gate_rows.dim() == 2 and gate_rows.shape[0] == n and 0 <= gate_col0
              and gate_col0 + o.shape[1] <= gate_rows.shape[1], "head_norm_gate: bad gate rows")
        gate_ptr, gate_stride, raw = (gate_rows.data_ptr() + 4 * int(gate_col0)), gate_rows.shape[1], GATE_ACTS[gate_act]
    _call("tp_head_norm_gate", _ptr(o), _ptr(weight), gate_ptr, float(eps), float(scale), _ptr(out), _dt(out),
          out.shape[1], int(out_col0), n, int(heads), vdim, per_head, int(gate_stride), raw, _stream())


def moe_plan(ids: torch.Tensor, experts: int):
    """Where every chosen (token, expert) pair goes when the pairs are brought into the order of the experts:
    ``ids`` int32 [n, top] -> (counts int32 [experts], offsets int32 [experts + 1], rank int32 [n, top]); pair (t, k)
    goes to row offsets[ids[t, k]] + rank[t, k], the pairs of one expert keeping the order of the tokens."""
    if _backend is not None:
        return _backend.moe_plan(ids, experts)
    _dev_ok(ids)
    _need(ids.dtype == torch.int32 and ids.dim() == 2, "moe_plan: ids must be int32 [n, top]")
    counts = torch.empty((experts,), dtype=torch.int32, device=ids.device)
    offsets = torch.empty((experts + 1,), dtype=torch.int32, device=ids.device)
    rank = torch.empty(ids.shape, dtype=torch.int32, device=ids.device)
    _call("tp_moe_plan", _ptr(ids), ids.shape[0], ids.shape[1], int(experts), _ptr(counts), _ptr(offsets), _ptr(rank), _stream())
    return counts, offsets, rank


def moe_linear_ok(experts: int, n: int, k: int, w, pairs: int = 0) -> bool:
    """Whether ``moe_linear`` takes the experts' stacked weight ``w`` (each [n, k]) and is the better way for ``pairs`` rows."""
    # (its tiles are 128 x 128 or 128 x 256; from some thousand rows an expert on, a product for each with tiles of 256 x 256 is the faster
    # product.  Both products of eight experts alone, 8,192 / 16,384 / 32,768 pairs, a product an expert against one launch: 4,096 x 4,096 gated
    # and 4,096 x 2,048 533 / 773 / 1,303 us against 439 / 827 / 1,831; 4,096 x 2,048 and 2,048 x 2,048 334 / 476 / 768 against 213 / 440 / 955; 7,168 x
    # 4,096 and 4,096 x 3,584 785 / 1,270 / 2,271 against 655 / 1,320 / 2,977.  But a product an expert waits on the host for the rows' counts and is
    # sixteen launches: the whole layer, routing and gathering included, 8,192 / 16,384 / 24,576 pairs at random, 744 / 1,236 / 1,593 us against 548 /
    # 1,070 / 1,489; 459 / 722 / 957 against 317 / 592 / 816; 1,050 / 1,638 / 2,320 against 828 / 1,615 / 2,331.  So up to 2,048 rows an expert go in one.)
    if pairs > 2048 * experts:
        return False
    return _backend is None and allow_mfma and w is not None and w.dtype == torch.bfloat16 and 0 < experts <= 64 and n % 16 == 0 and k % 64 == 0 and \
        tuple(w.shape) == (experts * n, k)


def moe_linear(x: torch.Tensor, w, offsets: torch.Tensor, experts: int, output: str = "float32") -> torch.Tensor:
    """bfloat16 rows sorted by expert (``moe_gather``; ``offsets`` int32 [experts + 1] of ``moe_plan``) times the stacked weights
    ``w`` [experts * n, k], a row with its expert's, in one launch and without the counts on the host.  ``output``: ``float32``
    [pairs, n]; ``swiglu``: bfloat16 [pairs, n / 2], the gated activation of interleaved gate/up rows; ``relu2``: bfloat16 [pairs, n],
    max(v, 0)^2.  Sizes: ``moe_linear_ok`` (``relu2``: n a multiple of 128)."""
    wd, wl = _w_args(w)
    _dev_ok(x, wd, offsets)
    pairs, k = x.shape
    n = w.shape[0] // experts
    _need(x.dtype == torch.bfloat16 and x.dim() == 2 and w.shape[1] == k and moe_linear_ok(experts, n, k, w), "moe_linear: bad operands")
    _i32(offsets, experts + 1, "offsets")
    mode = {"float32": 0, "swiglu": 2, "relu2": 3}[output]
    out = torch.empty((pairs, n // 2 if mode == 2 else n), dtype=torch.float32 if mode == 0 else torch.bfloat16, device=x.device)
    _call("tp_moe_linear", _ptr(x), _ptr(wd), int(bool(wl)), _ptr(out), mode, pairs, int(experts), _ptr(offsets), n, k, _stream(), tag=(pairs, n, k))
    return out


def moe_gather(x: torch.Tensor, ids: torch.Tensor, rank: torch.Tensor, offsets: torch.Tensor):
    """(rows [n * top, width] of ``x`` [n, width] in the order of the experts, row_of int32 [n, top]: the row of pair (t, k))."""
    if _backend is not None:
        return _backend.moe_gather(x, ids, rank, offsets)
    _dev_ok(x, ids, rank, offsets)
    n, top = ids.shape
    _need(x.dim() == 2 and x.shape[0] == n and (x.shape[1] * x.element_size()) % 4 == 0, "moe_gather: rows must be a multiple of four bytes")
    _need(rank.dtype == torch.int32 and tuple(rank.shape) == (n, top) and offsets.dtype == torch.int32, "moe_gather: bad plan")
    xg = torch.empty((n * top, x.shape[1]), dtype=x.dtype, device=x.device)
    row_of = torch.empty((n, top), dtype=torch.int32, device=x.device)
    _call("tp_moe_gather", _ptr(x), _ptr(ids), _ptr(rank), _ptr(offsets), _ptr(xg), _ptr(row_of), n, top, x.shape[1] * x.element_size(), _stream())
    return xg, row_of


def moe_scatter(yg: torch.Tensor, row_of: torch.Tensor, weights: torch.Tensor, y: Optional[torch.Tensor] = None) -> torch.Tensor:
    """y[t] (+)= sum_k weights[t, k] * yg[row_of[t, k]] (k ascending); ``y`` None: a new tensor."""
    if _backend is not None:
        return _backend.moe_scatter(yg, row_of, weights, y)
    _dev_ok(yg, row_of, weights, y)
    n, top = row_of.shape
    _need(yg.dtype == torch.float32 and yg.dim() == 2 and yg.shape[0] == n * top and weights.dtype == torch.float32
          and tuple(weights.shape) == (n, top) and row_of.dtype == torch.int32, "moe_scatter: bad operands")
    acc = y is not None
    if not acc:
        y = torch.empty((n, yg.shape[1]), dtype=torch.float32, device=yg.device)
    _need(y.dtype == torch.float32 and tuple(y.shape) == (n, yg.shape[1]), "moe_scatter: y must be float32 [n, width]")
    _call("tp_moe_scatter", _ptr(yg), _ptr(row_of), _ptr(weights), _ptr(y), n, top, yg.shape[1], int(acc), _stream())
    return y


def moe_spread(a: torch.Tensor, dense: torch.Tensor, experts: int) -> torch.Tensor:
    """``a`` [n, experts * ff] (all experts' activations of every row) -> [experts, n, ff]: each expert's activations
    as rows of its own, times the row's weight for the expert (``dense`` float32 [n, experts], zero where the expert
    was not chosen); the product is formed in float32 and rounded once."""
    if _backend is not None:
        return _backend.moe_spread(a, dense, experts)
    _dev_ok(a, dense)
    _need(a.dim() == 2 and a.shape[1] % experts == 0 and dense.dtype == torch.float32 and tuple(dense.shape) == (a.shape[0], experts),
          "moe_spread: bad operands")
    n, ff = a.shape[0], a.shape[1] // experts
    out = torch.empty((experts, n, ff), dtype=a.dtype, device=a.device)
    _call("tp_moe_spread", _ptr(a), _dt(a), _ptr(dense), _ptr(out), n, int(experts), ff, _stream())
    return out


# ---------------------------------------------------------------------------------
# Operations of layers with one norm for both sublayers, inputs convolved over time, a generalized delta rule, an
# attention over keys and values expanded from a latent, and a vector added to the stream between layers.

def rmsnorm_cols(x: torch.Tensor, col0: int, width: int, weight: torch.Tensor, eps: float, out_dtype: torch.dtype, groups: int = 1) -> torch.Tensor:
    """The RMS norm (in ``groups`` equal parts) of columns col0 .. col0 + width of float32 rows [n, wider], times
    ``weight`` [width] -> out_dtype [n, width]."""
    if _backend is not None:
        return _backend.rmsnorm_cols(x, col0, width, weight, eps, out_dtype, groups)
    _dev_ok(x, weight)
    _need(x.dtype == torch.float32 and x.dim() == 2 and 0 <= col0 and col0 + width <= x.shape[1], "rmsnorm_cols: bad rows")
    _need(weight.dtype == torch.float32 and weight.numel() == width and groups > 0 and width % groups == 0, "rmsnorm_cols: bad weight or groups")
    out = torch.empty((x.shape[0], width), dtype=out_dtype, device=x.device)
    _call("tp_group_rmsnorm", _ptr(x), int(x.shape[1]), int(col0), _ptr(weight), _ptr(None), _ptr(out), _dtcode(out_dtype),
          x.shape[0], int(width), int(groups), float(eps), _stream())
    return out


def residual_conv(x: torch.Tensor, weight: torch.Tensor, state: torch.Tensor, state_off: int, cu_seqlens: torch.Tensor,
                  token_req: torch.Tensor, state_slots: torch.Tensor, num_requests: int, out_dtype: torch.dtype, max_run: int = 0,
                  blocked=()):
    """What sublayers read of rows ``x`` (float32 [n, width]): for each of the ``weight`` [subs, taps, width] (tap-major,
    the last tap the current token's) x + conv(x) over each request's run of tokens, as ``out_dtype``; a list of
    ``subs`` tensors [n, width].  ``state`` float32 [slots, row]: from element ``state_off`` on a request's carried
    rows [taps - 1, width] (oldest first), read for the first tokens of a run and replaced by the run's last rows.  ``max_run``: the longest run
    (0: not known); runs of one token are one launch, which gives the sublayers named in ``blocked`` their rows as ``KBlocked``
    (``few_rows_ok``, at most four sublayers)."""
    if _backend is not None:
        return _backend.residual_conv(x, weight, state, state_off, cu_seqlens, token_req, state_slots, num_requests, out_dtype)
    _dev_ok(x, weight, state, cu_seqlens, token_req, state_slots)
    _need(x.dtype == torch.float32 and x.dim() == 2, "residual_conv: rows must be float32 [n, width]")
    n, width = x.shape
    _need(weight.dtype == torch.float32 and weight.dim() == 3 and weight.shape[2] == width, "residual_conv: weight must be float32 [subs, taps, width]")
    subs, taps = weight.shape[0], weight.shape[1]
    # (one tap carries nothing: a layer whose parts keep no state then has no state tensor)
    _need((state is None and taps == 1) or (state is not None and state.dtype == torch.float32 and state.dim() == 2 and state_off >= 0
                                            and state.shape[1] >= state_off + (taps - 1) * width), "residual_conv: state rows too short")
    _i32(cu_seqlens, num_requests + 1, "cu_seqlens")
    _i32(state_slots, num_requests, "state_slots")
    _i32(token_req, n, "token_req") if n else None
    out = torch.empty((subs, n, width), dtype=out_dtype, device=x.device)
    _call("tp_residual_conv", _ptr(x), _ptr(weight), _ptr(state), int(0 if state is None else state.shape[1]), int(state_off),
          _ptr(cu_seqlens), _ptr(token_req), _ptr(state_slots), _ptr(out), _dtcode(out_dtype), n, int(num_requests), width, taps, subs,
          int(max_run), sum(1 << i for i in blocked), _stream())
    return [KBlocked(out[i].view(width // 8, n, 8), n, width) if i in blocked else out[i] for i in range(subs)]


def norm_residual_conv_ok(n: int, width: int, groups: int, taps: int, subs: int, max_run: int) -> bool:
    """Whether ``norm_residual_conv`` takes a step of ``n`` tokens: single ones, few enough that a launch counts."""
    # (several parts: a row normed whole has a kernel that adds its squares in another order.  The gain grows with the rows, 128 of 4,096
    # 8.5 / 5.2 us; beyond 64 a launch no longer counts beside the products)
    return _backend is None and max_run == 1 and 0 < n <= 64 and groups > 1 and width % 8 == 0 and width % groups == 0 and width // groups % 4 == 0 and \
        width // groups <= 4096 and 2 <= taps <= 4 and 1 <= subs <= 2


def norm_residual_conv(h: torch.Tensor, norm_weight: torch.Tensor, eps: float, groups: int, weight: torch.Tensor, state: torch.Tensor,
                       state_off: int, token_req: torch.Tensor, state_slots: torch.Tensor, out_dtype: torch.dtype, blocked=()):
    """``residual_conv`` of the rows ``rmsnorm(h, norm_weight, eps, float32, groups=groups)`` in one launch, for runs of one token each
    (``norm_residual_conv_ok``), with the bits of the two."""
    _dev_ok(h, norm_weight, weight, state, token_req, state_slots)
    _need(h.dtype == torch.float32 and h.dim() == 2 and weight.dtype == torch.float32 and weight.dim() == 3 and weight.shape[2] == h.shape[1],
          "norm_residual_conv: rows must be float32 [n, width], weight float32 [subs, taps, width]")
    (n, width), (subs, taps) = h.shape, weight.shape[:2]
    _need(norm_residual_conv_ok(n, width, groups, taps, subs, 1), "norm_residual_conv: sizes")
    _need(norm_weight.dtype == torch.float32 and norm_weight.numel() == width, "norm_residual_conv: norm weight must be float32 [width]")
    _need(state.dtype == torch.float32 and state.dim() == 2 and state_off >= 0 and state.shape[1] >= state_off + (taps - 1) * width,
          "norm_residual_conv: state rows too short")
    _i32(token_req, n, "token_req")
    _need(state_slots.dtype == torch.int32, "state_slots must be int32")
    out = torch.empty((subs, n, width), dtype=out_dtype, device=h.device)
    _call("tp_norm_residual_conv", _ptr(h), _ptr(norm_weight), int(groups), float(eps), _ptr(weight), _ptr(state),
          int(state.shape[1]), int(state_off), _ptr(token_req), _ptr(state_slots), _ptr(out), _dtcode(out_dtype), n, width,
          taps, subs, sum(1 << i for i in blocked), _stream())
    return [KBlocked(out[i].view(width // 8, n, 8), n, width) if i in blocked else out[i] for i in range(subs)]


def add_row(h: torch.Tensor, table: torch.Tensor, row: int) -> None:
    """h[t] += table[row] for every row t, in place (float32)."""
    if _backend is not None:
        return _backend.add_row(h, table, row)
    _dev_ok(h, table)
    _need(h.dtype == torch.float32 and h.dim() == 2 and table.dtype == torch.float32 and table.dim() == 2 and table.shape[1] == h.shape[1]
          and 0 <= row < table.shape[0], "add_row: h float32 [n, width], table float32 [rows, width]")
    _call("tp_add_row", _ptr(h), (table.data_ptr() + 4 * int(row) * table.shape[1]), h.shape[0], h.shape[1], _stream())


def general_delta_scan(proj: torch.Tensor, col0: int, decay: torch.Tensor, a_bias: torch.Tensor, state: torch.Tensor, state_off: int,
                       cu_seqlens: torch.Tensor, state_slots: torch.Tensor, num_requests: int, heads: int, dim: int,
                       unit_eps: float) -> torch.Tensor:
    """The generalized delta rule per head over each request's run.  ``proj`` float32 rows hold, from column ``col0``
    on, r | k | v | a_raw, each [heads * dim]; a = sigmoid(a_raw + a_bias); ``decay`` float32 [n, heads * dim].  With the
    unit key u = k / sqrt(sum k^2 + unit_eps) and S [dim, dim] per head (kept at ``state[slot, state_off:]`` column by
    column):  S <- diag(decay) S - (a u) (u^T S) + k v^T (both terms read the old S);  o = S^T r.
    Returns o float32 [n, heads * dim]; the state is left as the run leaves it."""
    if _backend is not None:
        return _backend.general_delta_scan(proj, col0, decay, a_bias, state, state_off, cu_seqlens, state_slots, num_requests, heads, dim, unit_eps)
    _dev_ok(proj, decay, a_bias, state, cu_seqlens, state_slots)
    n, hd = proj.shape[0], heads * dim
    _need(proj.dtype == torch.float32 and proj.dim() == 2 and 0 <= col0 and col0 + 4 * hd <= proj.shape[1], "general_delta_scan: bad r | k | v | a rows")
    _need(decay.dtype == torch.float32 and tuple(decay.shape) == (n, hd), "general_delta_scan: decay must be float32 [n, heads * dim]")
    _need(a_bias.dtype == torch.float32 and a_bias.numel() == hd, "general_delta_scan: a_bias must be float32 [heads * dim]")
    _need(state.dtype == torch.float32 and state.dim() == 2 and state_off >= 0 and state.shape[1] >= state_off + hd * dim,
          "general_delta_scan: state rows too short")
    _i32(cu_seqlens, num_requests + 1, "cu_seqlens")
    _i32(state_slots, num_requests, "state_slots")
    y = torch.empty((n, hd), dtype=torch.float32, device=proj.device)
    scratch = torch.empty((max(1, n * 2 * hd + n * heads * 2),), dtype=torch.float32, device=proj.device)
    _call("tp_gdelta_scan", _ptr(proj), proj.shape[1], int(col0), _ptr(decay), _ptr(a_bias), _ptr(state), int(state.shape[1]),
          int(state_off), _ptr(cu_seqlens), _ptr(state_slots), _ptr(y), _ptr(scratch), n, int(num_requests), int(heads),
          int(dim), float(unit_eps), _stream())
    return y


def latent_rows(proj: torch.Tensor, q_col0: int, rot_col0: int, up: torch.Tensor, heads: int, dim: int, rot: int, vdim: int) -> torch.Tensor:
    """The rows q | k | v that ``rope_kv_write`` takes, for an attention whose keys and values are expanded from a
    latent: q [heads, rot + dim] is columns q_col0 .. of ``proj`` (float32 rows) as they stand; head h's key is the
    shared part proj[:, rot_col0 : rot_col0 + rot] followed by up[:, h * dim : (h + 1) * dim]; its value
    up[:, heads * dim + h * vdim : ...].  ``up`` float32 [n, >= heads * (dim + vdim)].  Returns float32
    [n, 2 * heads * (rot + dim) + heads * vdim]."""
    if _backend is not None:
        return _backend.latent_rows(proj, q_col0, rot_col0, up, heads, dim, rot, vdim)
    _dev_ok(proj, up)
    n = proj.shape[0]
    _need(proj.dtype == torch.float32 and proj.dim() == 2 and up.dtype == torch.float32 and up.dim() == 2 and up.shape[0] == n,
          "latent_rows: float32 rows")
    _need(0 <= q_col0 and q_col0 + heads * (rot + dim) <= proj.shape[1] and 0 <= rot_col0 and rot_col0 + rot <= proj.shape[1]
          and up.shape[1] >= heads * (dim + vdim), "latent_rows: rows too short")
    out = torch.empty((n, 2 * heads * (rot + dim) + heads * vdim), dtype=torch.float32, device=proj.device)
    _call("tp_latent_rows", _ptr(proj), int(proj.shape[1]), int(q_col0), int(rot_col0), _ptr(up), int(up.shape[1]),
          _ptr(out), n, int(heads), int(dim), int(rot), int(vdim), _stream())
    return out


def head_rmsnorm(rows: torch.Tensor, col_a: int, heads_a: int, weight_a: Optional[torch.Tensor], col_b: int, heads_b: int,
                 weight_b: Optional[torch.Tensor], dim: int, eps: float) -> None:
    """In place on float32 rows [n, wider]: each of the ``heads_a`` heads of ``dim`` columns from col_a on becomes
    x / sqrt(mean(x^2) + eps) * weight_a (float32 [dim], one for all heads), and likewise the ``heads_b`` heads from col_b
    on with weight_b (the queries and the keys of an attention in one launch)."""
    if _backend is not None:
        return _backend.head_rmsnorm(rows, col_a, heads_a, weight_a, col_b, heads_b, weight_b, dim, eps)
    _dev_ok(rows, weight_a, weight_b)
    _need(rows.dtype == torch.float32 and rows.dim() == 2, "head_rmsnorm: rows must be float32 [n, width]")
    for col, heads, w in ((col_a, heads_a, weight_a), (col_b, heads_b, weight_b)):
        _need(heads >= 0 and col >= 0 and col + heads * dim <= rows.shape[1], "head_rmsnorm: heads outside the rows")
        _need(heads == 0 or (w is not None and w.dtype == torch.float32 and w.numel() == dim), "head_rmsnorm: weight must be float32 [dim]")
    _call("tp_head_rmsnorm", _ptr(rows), int(rows.shape[1]), int(col_a), int(heads_a), _ptr(weight_a), int(col_b), int(heads_b),
          _ptr(weight_b), int(dim), float(eps), rows.shape[0], _stream())


def vector_store(c: torch.Tensor, slots: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor) -> None:
    """One vector a token, ``c`` [n, dim], into cache place ``slots`` of keys [pages, 1, page_size, dim] and of transposed
    values [pages, 1, dim, page_size] (an attention whose keys are its values reads both)."""
    if _backend is not None:
        return _backend.vector_store(c, slots, k_cache, v_cache)
    _dev_ok(c, slots, k_cache, v_cache)
    _need(c.dim() == 2 and k_cache.dim() == 4 and v_cache.dim() == 4 and k_cache.shape[1] == 1, "vector_store: bad operand ranks")
    n, dim = c.shape
    pages, _, page_size, d2 = k_cache.shape
    _need(d2 == dim and tuple(v_cache.shape) == (pages, 1, dim, page_size), "vector_store: caches must be k [pages, 1, page_size, dim], v [pages, 1, dim, page_size]")
    _need(c.dtype == k_cache.dtype == v_cache.dtype, "vector_store: vector and cache types differ")
    _i32(slots, n, "slots") if n else None
    _call("tp_vector_store", _ptr(c), _dt(c), _ptr(slots), _ptr(k_cache), _ptr(v_cache), n, dim, page_size, _stream())


def latent_norms_ok(rows: torch.Tensor, q_col0: int, q_dim: int, c_col0: int, c_dim: int, cache_dtype: torch.dtype, dtype: torch.dtype) -> bool:
    """Whether ``latent_norms`` takes these rows: few of them (a launch counts), both parts in 16-byte pieces and one type for all results."""
    return _backend is None and 0 < rows.shape[0] <= 64 and dtype == cache_dtype and rows.shape[1] % 4 == 0 and rows.is_contiguous() and \
        rows.data_ptr() % 16 == 0 and all(v % 4 == 0 for v in (q_col0, q_dim, c_col0, c_dim)) and 0 < q_dim <= 4096 and 0 < c_dim <= 4096 and \
        c_dim * dtype.itemsize % 16 == 0 and q_dim * dtype.itemsize % 16 == 0


def latent_norms(rows: torch.Tensor, q_col0: int, q_dim: int, q_weight: torch.Tensor, c_col0: int, c_dim: int, c_weight: torch.Tensor, eps: float,
                 slots: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor) -> torch.Tensor:
    """``vector_store(rmsnorm_cols(rows, c_col0, c_dim, c_weight, eps, k_cache.dtype), slots, k_cache, v_cache)`` and the returned
    ``rmsnorm_cols(rows, q_col0, q_dim, q_weight, eps, k_cache.dtype)`` in one launch (``latent_norms_ok``), with their bits."""
    _dev_ok(rows, q_weight, c_weight, slots, k_cache, v_cache)
    _need(rows.dtype == torch.float32 and rows.dim() == 2 and latent_norms_ok(rows, q_col0, q_dim, c_col0, c_dim, k_cache.dtype, k_cache.dtype)
          and 0 <= q_col0 and q_col0 + q_dim <= rows.shape[1] and 0 <= c_col0 and c_col0 + c_dim <= rows.shape[1], "latent_norms: bad rows")
    for w, d in ((q_weight, q_dim), (c_weight, c_dim)):
        _need(w.dtype == torch.float32 and w.numel() == d, "latent_norms: weights must be float32, one for each column")
    _need(k_cache.dim() == 4 and k_cache.shape[1] == 1 and k_cache.shape[3] == c_dim and v_cache.dtype == k_cache.dtype
          and tuple(v_cache.shape) == (k_cache.shape[0], 1, c_dim, k_cache.shape[2]),
          "latent_norms: caches must be k [pages, 1, page_size, dim], v [pages, 1, dim, page_size]")
    n = rows.shape[0]
    _i32(slots, n, "slots")
    cq = torch.empty((n, q_dim), dtype=k_cache.dtype, device=rows.device)
    _call("tp_latent_norms", _ptr(rows), int(rows.shape[1]), int(q_col0), int(q_dim), _ptr(q_weight), int(c_col0), int(c_dim),
          _ptr(c_weight), float(eps), _ptr(cq), _ptr(slots), _ptr(k_cache), _ptr(v_cache), _dt(k_cache), n, k_cache.shape[2], _stream())
    return cq


def mlstm_scan(proj: torch.Tensor, col0: int, i_bias: torch.Tensor, f_bias: torch.Tensor, cap: float, q_scale: float,
               state: torch.Tensor, state_off: int, cu_seqlens: torch.Tensor, state_slots: torch.Tensor, num_requests: int,
               heads: int, dim: int, vdim: int, norm_weight: torch.Tensor, eps: float, scale: float, out: torch.Tensor,
               out_col0: int) -> None:
    """The matrix-memory recurrence of an mLSTM mixer over each request's run of tokens, and its read-out as the rows
    of the output product.  ``proj`` float32 [n, wider] holds from col0 on [q | k | v | gate | i | f] (heads * dim,
    heads * dim, heads * vdim, heads * vdim, heads, heads columns).  With i = cap tanh((x_i + i_bias) / cap) and
    f = logsigmoid(cap tanh((x_f + f_bias) / cap)) per head: m' = max(f + m, i); S' = e^(f + m - m') S + e^(i - m') k v^T;
    n' likewise with k alone; o = S'^T (q * q_scale) / (max(|n' . q|, e^(-m')) + 1e-6).  Then per head o over its root
    mean square (``eps``), times ``norm_weight`` [heads * vdim], times sigmoid(gate), times ``scale``, into columns
    out_col0 .. of ``out``.  A request's state (float32 row of ``state`` from state_off on, heads * (vdim + 1) * (dim + 1)
    numbers: per head the memory column by column with n as the last column, then a copy of m per column) is read and
    left updated."""
    if _backend is not None:
        return _backend.mlstm_scan(proj, col0, i_bias, f_bias, cap, q_scale, state, state_off, cu_seqlens, state_slots, num_requests,
                                   heads, dim, vdim, norm_weight, eps, scale, out, out_col0)
    _dev_ok(proj, i_bias, f_bias, state, cu_seqlens, state_slots, norm_weight, out)
    _need(proj.dtype == torch.float32 and proj.dim() == 2, "mlstm_scan: rows must be float32 [n, width]")
    n = proj.shape[0]
    width = 2 * heads * dim + 2 * heads * vdim + 2 * heads
    _need(0 <= col0 and col0 + width <= proj.shape[1], "mlstm_scan: rows too short")
    for b in (i_bias, f_bias):
        _need(b.dtype == torch.float32 and b.numel() == heads, "mlstm_scan: gate biases must be float32 [heads]")
    _need(norm_weight.dtype == torch.float32 and norm_weight.numel() == heads * vdim, "mlstm_scan: norm weight must be float32 [heads * vdim]")
    _need(state.dtype == torch.float32 and state.dim() == 2 and state.shape[1] >= state_off + heads * (vdim + 1) * (dim + 1),
          "mlstm_scan: state rows too short")
    _i32(cu_seqlens, num_requests + 1, "cu_seqlens")
    _i32(state_slots, num_requests, "state_slots")
    _need(out.dim() == 2 and out.shape[0] == n and 0 <= out_col0 and out_col0 + heads * vdim <= out.shape[1], "mlstm_scan: output rows too short")
    scratch = torch.empty((max(2, n * heads * (vdim + 4)),), dtype=torch.float32, device=proj.device)
    _call("tp_mlstm_scan", _ptr(proj), proj.shape[1], int(col0), _ptr(i_bias), _ptr(f_bias), float(cap), float(q_scale),
          _ptr(state), int(state.shape[1]), int(state_off), _ptr(cu_seqlens), _ptr(state_slots), _ptr(scratch),
          _ptr(norm_weight), float(eps), float(scale), _ptr(out), _dt(out), out.shape[1], int(out_col0), n,
          int(num_requests), int(heads), int(dim), int(vdim), _stream())


# ---------------------------------------------------------------------------------
# Operations of mixers around a linear recurrence: mixes of a row and the row before it, and the recurrence.

def token_shift(x: torch.Tensor, mu: torch.Tensor, state: torch.Tensor, state_off: int, cu_seqlens: torch.Tensor, token_req: torch.Tensor,
                state_slots: torch.Tensor, num_requests: int, out_dtype: torch.dtype, max_run: Optional[int] = None,
                blocked: bool = False):
    """Mixes of float32 rows ``x`` [n, width] with the rows before them in their requests: for each of the ``mu`` [mixes,
    width] x + (x' - x) * mu, as ``out_dtype``; a list of tensors [n, width].  x' of a run's first token is what the request's
    state holds (``state`` float32 [slots, row], ``width`` numbers from ``state_off`` on); the run's last row is left there.
    ``max_run``: the longest run of the step (None: unknown).  ``blocked``: one tensor [mixes, width / 8, n, 8] instead (what
    ``group_linear`` takes)."""
    if _backend is not None:
        return _backend.token_shift(x, mu, state, state_off, cu_seqlens, token_req, state_slots, num_requests, out_dtype)
    _dev_ok(x, mu, state, cu_seqlens, token_req, state_slots)
    _need(x.dtype == torch.float32 and x.dim() == 2, "token_shift: rows must be float32 [n, width]")
    n, width = x.shape
    _need(mu.dtype == torch.float32 and mu.dim() == 2 and mu.shape[1] == width, "token_shift: mu must be float32 [mixes, width]")
    _need(state.dtype == torch.float32 and state.dim() == 2 and state_off >= 0 and state.shape[1] >= state_off + width, "token_shift: state rows too short")
    _i32(cu_seqlens, num_requests + 1, "cu_seqlens")
    _i32(state_slots, num_requests, "state_slots")
    _i32(token_req, n, "token_req") if n else None
    mixes = mu.shape[0]
    out = torch.empty((mixes, width // 8, n, 8) if blocked else (mixes, n, width), dtype=out_dtype, device=x.device)
    _call("tp_token_shift", _ptr(x), _ptr(mu), _ptr(state), int(state.shape[1]), int(state_off), _ptr(cu_seqlens),
          _ptr(token_req), _ptr(state_slots), _ptr(out), _dtcode(out_dtype), n, int(num_requests), width, mixes, int(max_run == 1), int(blocked), _stream())
    return out if blocked else list(out.unbind(0))


#: runs longer than a piece are cut into pieces that run side by side; a piece has at least this many tokens
scan_min_piece = 64
#: and is lengthened while the pieces of a step make more blocks than this
scan_target_blocks = 1024


def scan_piece(n: int, max_run: int, heads: int, dim: int, vdim: int) -> int:
    """Tokens of a piece of ``linear_scan`` (0: runs are not cut)."""
    if dim > 128:
        return 0
    blocks = heads * max(1, vdim // 64)
    piece = max(scan_min_piece, -(-n * blocks // scan_target_blocks))
    piece = -(-piece // 16) * 16
    return 0 if max_run <= piece else piece


def linear_scan(q, k, v, decay: torch.Tensor, state: torch.Tensor, state_off: int, cu_seqlens: torch.Tensor, state_slots: torch.Tensor,
                num_requests: int, heads: int, dim: int, vdim: int, bonus: Optional[torch.Tensor] = None, q_scale: float = 1.0,
                max_run: Optional[int] = None) -> torch.Tensor:
    """The recurrence S <- diag(decay) S + k v^T per head over each request's run of tokens.  ``q``, ``k`` and ``v`` are pairs
    (float32 rows [n, wider], first column) of heads * dim, heads * dim and heads * vdim columns; ``decay`` float32 [n,
    heads * dim].  Without ``bonus`` a token reads behind its update, o = S^T (q * q_scale); with it (float32 [heads *
    dim]) in front of it, o = (S + diag(bonus) k v^T)^T (q * q_scale).  S [dim, vdim] per head lies at ``state[slot,
    state_off:]`` column by column, [heads, vdim, dim], and is left as the run leaves it.  ``max_run``: the longest run of the
    step (None: the step's tokens).  Returns o float32 [n, heads * vdim]."""
    if _backend is not None:
        return _backend.linear_scan(q, k, v, decay, state, state_off, cu_seqlens, state_slots, num_requests, heads, dim, vdim, bonus, q_scale)
    n = decay.shape[0]
    _dev_ok(q[0], k[0], v[0], decay, state, cu_seqlens, state_slots, bonus)
    for (rows, col), width, what in ((q, heads * dim, "q"), (k, heads * dim, "k"), (v, heads * vdim, "v")):
        if not (rows.dtype == torch.float32 and rows.dim() == 2 and rows.shape[0] == n and 0 <= col and col + width <= rows.shape[1]):
            raise KernelError(f"linear_scan: bad {what} rows")
    _need(decay.dtype == torch.float32 and tuple(decay.shape) == (n, heads * dim), "linear_scan: decay must be float32 [n, heads * dim]")
    _need(bonus is None or (bonus.dtype == torch.float32 and bonus.numel() == heads * dim), "linear_scan: bonus must be float32 [heads * dim]")
    _need(state.dtype == torch.float32 and state.dim() == 2 and state_off >= 0 and state.shape[1] >= state_off + heads * dim * vdim,
          "linear_scan: state rows too short")
    _i32(cu_seqlens, num_requests + 1, "cu_seqlens")
    _i32(state_slots, num_requests, "state_slots")
    max_run = n if max_run is None else int(max_run)
    y = torch.empty((n, heads * vdim), dtype=torch.float32, device=decay.device)
    piece, scratch, pieces = scan_piece(n, max_run, heads, dim, vdim), None, 0
    if piece:
        # (a request's pieces start at place cu_seqlens[r] // piece + r of the scratch)
        pieces = n // piece + num_requests
        scratch = torch.empty((pieces * heads * dim * (vdim + 1),), dtype=torch.float32, device=decay.device)
    at = lambda rows: (rows[0].data_ptr() + 4 * int(rows[1]))
    _call("tp_linear_scan", at(q), q[0].shape[1], at(k), k[0].shape[1], at(v), v[0].shape[1], _ptr(decay), _ptr(bonus), float(q_scale),
          _ptr(state), int(state.shape[1]), int(state_off), _ptr(cu_seqlens), _ptr(state_slots), _ptr(y), n,
          int(num_requests), int(heads), int(dim), int(vdim), max_run, piece, pieces, _ptr(scratch), _stream())
    return y


# ---------------------------------------------------------------------------------
# One token a request through a whole recurrent mixer.

#: steps of up to this many requests take a recurrent mixer as one launch (0: never): up to 64 with the bits of the separate kernels,
#: beyond, where ``lowrank_up`` adds its products in another order, with the same rounding
mixer_step_rows = 128


def mixer_step_ok(n: int, max_run: int, heads: int, dim: int, vdim: int, ranks, state: torch.Tensor, state_off: int, out: torch.Tensor, out_col0: int,
                  gate_col0: int = 0, gate_width: int = 0) -> bool:
    """Whether the one-launch steps below take ``n`` requests of ``max_run`` tokens each, at most: ``heads`` heads of ``dim`` by
    ``vdim`` elements, low-rank projections of ``ranks``, the head's state at ``state_off`` of the rows of ``state``, results from
    column ``out_col0`` of ``out``, a raw gate from column ``gate_col0`` of rows ``gate_width`` wide."""
    # (a head's block has a fixed part that a small state does not pay for once there are more than four blocks a CU: 64 heads of
    # 64 x 64, a captured chain, separate kernels / one launch: 8 requests 12.8 / 9.0 us, 16: 17.3 / 15.5, 64: 44 / 53; 32 heads of
    # 128 x 128, 8 requests 26 / 14 us, 64: 85 / 68, 128: 205 / 154)
    if dim * vdim < 8192 and n * heads > 1024:
        return False
    return _backend is None and max_run == 1 and 0 < n <= mixer_step_rows and 32 < dim <= 128 and dim % 4 == 0 and 0 < vdim <= 128 and \
        vdim % 4 == 0 and all(0 < r <= 128 for r in ranks) and state.shape[1] % 4 == 0 and state_off % 4 == 0 and state.data_ptr() % 16 == 0 and \
        out.shape[1] % 4 == 0 and out_col0 % 4 == 0 and out.data_ptr() % 16 == 0 and gate_col0 % 4 == 0 and gate_width % 4 == 0


def _step_state(n, state, token_req, state_slots, out, out_col0, columns, what):
    if not (state.dtype == torch.float32 and state.dim() == 2 and out.dim() == 2 and out.shape[0] == n and 0 <= out_col0
            and out_col0 + columns <= out.shape[1]):
        raise KernelError(f"{what}: bad state or output rows")
    _i32(token_req, n, "token_req")
    _i32(state_slots, n, "state_slots")


def step_buffer():
    """Host memory for a step that is written down (``prepared``)."""
    return ctypes.create_string_buffer(int(library().tp_step_prepared_size()))


def delta_step(proj: torch.Tensor, col0: int, beta_col0: int, a_col0: int, g_col0: int, conv_w: torch.Tensor, a2_t: torch.Tensor,
               g2_t: torch.Tensor, a_log: torch.Tensor, dt_bias: torch.Tensor, norm_w: torch.Tensor, state: torch.Tensor, conv_off: int,
               state_off: int, token_req: torch.Tensor, state_slots: torch.Tensor, heads: int, dim: int, vdim: int, q_scale: float,
               unit_eps: float, norm_eps: float, scale: float, out: torch.Tensor, out_col0: int, prepared=None) -> None:
    """One token a request of a gated delta rule with as many key heads as heads: ``causal_conv`` (with SiLU) over the columns
    q | k | v from ``col0`` on, ``lowrank_up`` for the decay and the gate, ``delta_scan`` and ``head_norm_gate``, in one launch and
    with the same bits (``mixer_step_ok`` says for which sizes).  ``prepared`` (``step_buffer()``): the step is written down there for
    ``attention_rows`` instead of launched; its tensors have to live until that call."""
    _dev_ok(proj, conv_w, a2_t, g2_t, a_log, dt_bias, norm_w, state, token_req, state_slots, out)
    n, taps = proj.shape[0], conv_w.shape[0]
    _step_state(n, state, token_req, state_slots, out, out_col0, heads * vdim, "delta_step")
    _need(proj.dtype == torch.float32 and proj.dim() == 2 and col0 >= 0 and col0 + heads * (2 * dim + vdim) <= proj.shape[1]
          and 0 <= beta_col0 and beta_col0 + heads <= proj.shape[1] and 0 <= a_col0 and a_col0 + a2_t.shape[0] <= proj.shape[1]
          and 0 <= g_col0 and g_col0 + g2_t.shape[0] <= proj.shape[1], "delta_step: bad projection rows")
    _need(conv_w.dtype == a2_t.dtype == g2_t.dtype == a_log.dtype == dt_bias.dtype == norm_w.dtype == torch.float32
          and conv_w.shape[1] == heads * (2 * dim + vdim) and a2_t.shape[1] == heads * dim and g2_t.shape[1] == heads * vdim
          and a_log.numel() == heads and dt_bias.numel() == heads * dim and norm_w.numel() == vdim, "delta_step: bad weights")
    _call("tp_delta_step", _ptr(proj), int(proj.shape[1]), int(col0), int(beta_col0), int(a_col0), a2_t.shape[0], int(g_col0),
          g2_t.shape[0], _ptr(conv_w), taps, _ptr(a2_t), _ptr(g2_t), _ptr(a_log), _ptr(dt_bias), _ptr(norm_w), _ptr(state),
          int(state.shape[1]), int(conv_off), int(state_off), _ptr(token_req), _ptr(state_slots), _ptr(out),
          _dt(out), int(out.shape[1]), int(out_col0), n, int(heads), int(dim), int(vdim), float(q_scale),
          float(unit_eps), float(norm_eps), float(scale), prepared, _stream())


def general_delta_step(proj: torch.Tensor, col0: int, gate_col0: int, w_col0: int, w2_t: torch.Tensor, w0: torch.Tensor, rate: float,
                       a_bias: torch.Tensor, norm_w: torch.Tensor, state: torch.Tensor, state_off: int, token_req: torch.Tensor,
                       state_slots: torch.Tensor, heads: int, dim: int, unit_eps: float, norm_eps: float, scale: float, out: torch.Tensor,
                       out_col0: int) -> None:
    """One token a request of a generalized delta rule: ``lowrank_up`` for the decay, ``general_delta_scan`` and
    ``head_norm_gate`` with the raw gate columns, in one launch and with the same bits."""
    _dev_ok(proj, w2_t, w0, a_bias, norm_w, state, token_req, state_slots, out)
    n, hd = proj.shape[0], heads * dim
    _step_state(n, state, token_req, state_slots, out, out_col0, hd, "general_delta_step")
    _need(proj.dtype == torch.float32 and proj.dim() == 2 and col0 >= 0 and col0 + 4 * hd <= proj.shape[1] and 0 <= gate_col0
          and gate_col0 + hd <= proj.shape[1] and 0 <= w_col0 and w_col0 + w2_t.shape[0] <= proj.shape[1], "general_delta_step: bad projection rows")
    _need(w2_t.dtype == w0.dtype == a_bias.dtype == norm_w.dtype == torch.float32 and w2_t.shape[1] == hd and w0.numel() == hd
          and a_bias.numel() == hd and norm_w.numel() == hd, "general_delta_step: bad weights")
    _call("tp_general_delta_step", _ptr(proj), int(proj.shape[1]), int(col0), int(gate_col0), int(w_col0), w2_t.shape[0], _ptr(w2_t),
          _ptr(w0), float(rate), _ptr(a_bias), _ptr(norm_w), _ptr(state), int(state.shape[1]), int(state_off),
          _ptr(token_req), _ptr(state_slots), _ptr(out), _dt(out), int(out.shape[1]), int(out_col0), n, int(heads), int(dim),
          float(unit_eps), float(norm_eps), float(scale), _stream())


def linear_step(q, k, v, x, w2_t: torch.Tensor, mode: str, bias: torch.Tensor, rate: float, in_act: Optional[str],
                bonus: Optional[torch.Tensor], q_scale: float, gate, norm_w: torch.Tensor, norm_eps: float, scale: float, state: torch.Tensor,
                state_off: int, token_req: torch.Tensor, state_slots: torch.Tensor, heads: int, dim: int, vdim: int, out: torch.Tensor,
                out_col0: int, prepared=None) -> None:
    """One token a request of a linear recurrence: ``lowrank_up`` (``mode`` of rows ``x``) for the decay, ``linear_scan`` and
    ``head_norm_gate`` with the SiLU of the raw gate columns, in one launch and with the same bits.  ``q``, ``k``, ``v``, ``x`` and
    ``gate`` are pairs (float32 rows, first column).  ``prepared``: as of ``delta_step``."""
    _need(mode in ("rate_sigmoid", "exp_exp", "root_sigmoid") and in_act in (None, "tanh"), "linear_step: bad decay")
    _dev_ok(q[0], k[0], v[0], x[0], gate[0], w2_t, bias, bonus, norm_w, state, token_req, state_slots, out)
    n = q[0].shape[0]
    _step_state(n, state, token_req, state_slots, out, out_col0, heads * vdim, "linear_step")
    for (rows, col), width, what in ((q, heads * dim, "q"), (k, heads * dim, "k"), (v, heads * vdim, "v"), (x, w2_t.shape[0], "decay"),
                                     (gate, heads * vdim, "gate")):
        if not (rows.dtype == torch.float32 and rows.dim() == 2 and rows.shape[0] == n and 0 <= col and col + width <= rows.shape[1]):
            raise KernelError(f"linear_step: bad {what} rows")
    _need(w2_t.dtype == bias.dtype == norm_w.dtype == torch.float32 and w2_t.shape[1] == heads * dim and bias.numel() == heads * dim
          and norm_w.numel() in (vdim, heads * vdim) and (bonus is None or (bonus.dtype == torch.float32 and bonus.numel() == heads * dim)),
          "linear_step: bad weights")
    at = lambda rows: (rows[0].data_ptr() + 4 * int(rows[1]))
    wide = lambda rows: int(rows[0].shape[1])
    _call("tp_linear_step", at(q), wide(q), at(k), wide(k), at(v), wide(v), at(x), wide(x), w2_t.shape[0], _ptr(w2_t), _ptr(bias),
          LOWRANK_MODES[mode], 1 if in_act == "tanh" else 0, float(rate), _ptr(bonus), float(q_scale), at(gate), wide(gate),
          GATE_ACTS["silu"], _ptr(norm_w), int(norm_w.numel() == heads * vdim and heads > 1), _ptr(state), int(state.shape[1]),
          int(state_off), _ptr(token_req), _ptr(state_slots), _ptr(out), _dt(out), int(out.shape[1]), int(out_col0), n,
          int(heads), int(dim), int(vdim), float(norm_eps), float(scale), prepared, _stream())


# ---------------------------------------------------------------------------------
# Products of decode steps that come in groups.

def few_rows_ok(m: int, width: int, dtype: torch.dtype) -> bool:
    """Whether ``m`` rows of that width are few enough for the products that read them k-blocked."""
    return _backend is None and allow_mfma and dtype == torch.bfloat16 and 0 < m <= 16 and width % 64 == 0


def block_rows(x: torch.Tensor) -> KBlocked:
    """bfloat16 rows [m, k] as ``KBlocked``."""
    _dev_ok(x)
    _need(x.dtype == torch.bfloat16 and x.dim() == 2 and x.shape[1] % 8 == 0, "block_rows: rows must be bfloat16 [m, a multiple of eight]")
    m, k = x.shape
    out = torch.empty((k // 8, m, 8), dtype=x.dtype, device=x.device)
    _call("tp_block_rows", _ptr(x), _ptr(out), m, k, _stream())
    return KBlocked(out, m, k)


def group_linear_ok(m: int, w) -> bool:
    """Whether ``group_linear`` takes ``m`` rows and the stacked weight."""
    return isinstance(w, TiledWeight) and few_rows_ok(m, w.shape[1], w.dtype)


def group_linear(x: torch.Tensor, w, ends) -> torch.Tensor:
    """Several products of at most 16 bfloat16 rows in one launch: ``x`` [groups, k / 8, m, 8] (k-blocked), ``w`` the tiled
    weights [n, k] of all groups stacked, group g's rows ending at ``ends[g]`` (multiples of 16).  Float32 [m, n]."""
    _need(isinstance(w, TiledWeight) and x.dim() == 4 and x.dtype == torch.bfloat16 and x.shape[3] == 8, "group_linear: k-blocked rows and tiled weights")
    groups, k8, m, _ = x.shape
    n, k = w.shape
    _dev_ok(x, w.data)
    _need(k == 8 * k8 and len(ends) == groups and ends[-1] == n, "group_linear: groups and weight disagree")
    out = torch.empty((m, n), dtype=torch.float32, device=x.device)
    _call("tp_group_linear", _ptr(x), _ptr(w.data), _ptr(out), (ctypes.c_int * groups)(*ends), groups, m, n, k, _stream(), tag=(m, n, k))
    return out


def moe_few_ok(m: int, experts: int, ff: int, w_up, w_down) -> bool:
    """Whether ``moe_few`` takes ``m`` rows and these stacked experts."""
    return (isinstance(w_up, TiledWeight) and isinstance(w_down, TiledWeight) and experts <= 512 and ff % 64 == 0
            and few_rows_ok(m, w_up.shape[1], w_up.dtype))


def moe_open_ok(experts: int, w_router, k: int, w_shared_up=None, w_shared_down=None, size: int = 0) -> bool:
    """Whether ``moe_open`` takes this router and, if there is one, this shared expert (of ``size``, without a gated activation)."""
    if not (isinstance(w_router, TiledWeight) and experts <= 64 and w_router.shape[0] == -(-experts // 16) * 16 and k % 64 == 0):
        return False
    return w_shared_up is None or (isinstance(w_shared_up, TiledWeight) and isinstance(w_shared_down, TiledWeight) and size % 64 == 0)


def moe_open(x: KBlocked, w_router, correction: Optional[torch.Tensor], experts: int, top: int, groups: int, keep: int, score: str = "softmax",
             group_best: int = 1, normalize: bool = False, sum_eps: float = 0.0, scale: float = 1.0, bias: Optional[torch.Tensor] = None,
             shared: Optional[tuple] = None):
    """The router of at most 16 rows in one launch: ``moe_route`` of the rows' product with the tiled ``w_router`` (its rows padded to 16),
    the same bits.  ``shared`` = (tiled up weight, size, activation, whether its row ``size`` is a gate's): the shared expert's up product
    beside it.  Returns (dense, ids, weights, (activated rows bfloat16 [size / 8, m, 8], raw gate float32 [m] or None) or None)."""
    m, k = x.shape
    _dev_ok(x.data, w_router.data, correction, bias)
    _need(moe_open_ok(experts, w_router, k) and w_router.shape[1] == k and score in ROUTE_SCORES and group_best >= 1, "moe_open: sizes that it does not take")
    _need(bias is None or (bias.dtype == torch.float32 and bias.numel() == experts), "moe_open: bias must be float32 [experts]")
    _need(correction is None or (correction.dtype == torch.float32 and correction.numel() == experts), "moe_open: correction must be float32 [experts]")
    dev = x.data.device
    dense = torch.empty((m, experts), dtype=torch.float32, device=dev)
    ids = torch.empty((m, top), dtype=torch.int32, device=dev)
    weights = torch.empty((m, top), dtype=torch.float32, device=dev)
    w_shared, size, kind, a, gate = None, 0, 0, None, None
    if shared is not None:
        w_shared, size, activation, gated = shared
        _dev_ok(w_shared.data)
        _need(w_shared.shape[1] == k and size + int(gated) <= w_shared.shape[0], "moe_open: bad shared expert")
        kind = ACTIVATIONS[activation]
        a = torch.empty((size // 8, m, 8), dtype=torch.bfloat16, device=dev)
        gate = torch.empty((m,), dtype=torch.float32, device=dev) if gated else None
    _call("tp_moe_open", _ptr(x.data), _ptr(w_router.data), _ptr(correction), _ptr(bias), int(experts), int(top), int(groups), int(keep), _ptr(dense),
          _ptr(ids), _ptr(weights), m, k, ROUTE_SCORES[score], int(group_best), int(bool(normalize)), float(sum_eps), float(scale),
          _ptr(None if w_shared is None else w_shared.data), 0 if w_shared is None else w_shared.shape[0], int(size), kind, _ptr(a), _ptr(gate), _stream())
    return dense, ids, weights, None if shared is None else (a, gate)


def moe_few(x: KBlocked, w_up, w_down, dense: torch.Tensor, ff: int, activation: Optional[str], y: Optional[torch.Tensor] = None,
            shared: Optional[tuple] = None, partial_ok: bool = False):
    """The routed experts of at most 16 rows: y (+)= sum_e down_e(f(up_e x) * dense[:, e]), skipping the weights of experts
    whose column of ``dense`` (float32 [m, experts]) is zero.  ``w_up``: the experts' tiled up weights stacked
    ([experts * ff, k]; ``activation`` None: gate and up rows interleaved by eights, [2 experts * ff, k], f = silu(gate) * up);
    ``w_down``: their tiled [n, ff] one behind the other, as a ``TiledWeight`` of [experts * n, ff].  ``y`` float32 [m, n] or None.
    ``shared`` = (tiled down weight [n, size], activated rows, raw gate or None, as of ``moe_open``): the shared expert's output behind
    the routed sum, times sigmoid(gate).  With ``partial_ok`` and no ``y`` the result may be ``Partials`` (``few_splits``)."""
    m, k = x.shape
    experts = dense.shape[1]
    w_s, a_s, gate = shared if shared is not None else (None, None, None)
    n = w_down.shape[0] // experts
    _dev_ok(x.data, w_up.data, w_down.data, dense, y)
    rows = ff if activation is not None else 2 * ff
    _need(tuple(w_up.shape) == (experts * rows, k) and tuple(w_down.shape) == (experts * n, ff), "moe_few: weights disagree with the sizes")
    _need(dense.dtype == torch.float32 and tuple(dense.shape) == (m, experts), "moe_few: dense must be float32 [m, experts]")
    _need(y is None or (y.dtype == torch.float32 and tuple(y.shape) == (m, n)), "moe_few: y must be float32 [m, n]")
    if w_s is not None:
        _dev_ok(w_s.data, a_s, gate)
        _need(w_s.shape[0] == n and tuple(a_s.shape) == (w_s.shape[1] // 8, m, 8) and a_s.dtype == torch.bfloat16 and
              (gate is None or (gate.dtype == torch.float32 and gate.numel() == m)), "moe_few: shared expert disagrees with the sizes")
    acc = y is not None
    # (an expert's own K is what is cut, so that a row's sums do not depend on the experts of the rows beside it; whole turns of eight runs)
    parts = 1
    while partial_ok and not acc and parts < 4 and 2 * parts * (n // 16) <= 256 and ff % (2048 * parts) == 0 and \
            (w_s is None or w_s.shape[1] % (64 * parts) == 0):
        parts *= 2
    if not acc:
        y = torch.empty((parts, m, n) if parts > 1 else (m, n), dtype=torch.float32, device=dense.device)
    a = torch.empty((experts * ff // 8, m, 8), dtype=torch.bfloat16, device=dense.device)
    _call("tp_moe_few", _ptr(x.data), _ptr(w_up.data), _ptr(w_down.data), _ptr(dense), _ptr(a), _ptr(y), m, experts, int(ff), k, n,
          int(activation is None), 0 if activation is None else ACTIVATIONS[activation], int(acc), _ptr(None if w_s is None else w_s.data), _ptr(a_s),
          _ptr(gate), 0 if w_s is None else w_s.shape[1], parts, _stream(), tag=(m, experts, ff, k))
    return y if parts == 1 else Partials(y)
