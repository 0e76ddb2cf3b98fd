"""Python face of the HIP kernels: shape checks on the host, then one C call per kernel.

There is no other implementation behind these functions: without a GPU, or
without the compiled library, they raise.  Tensors are torch tensors on the
GPU; torch serves as the allocator and, for large bfloat16 matrix products,
as the door to the vendor's GEMM library (the reference uses cuBLAS there,
`candle-core/src/cuda_backend/mod.rs:2260-2305`).
"""
from __future__ import annotations

import ctypes
import functools
import os
from typing import Dict, Optional, Sequence, Tuple

import torch

from . import build as _build

F32, BF16 = 0, 1
_DT = {torch.float32: F32, torch.bfloat16: BF16}


class KernelError(RuntimeError):
    pass


_LIBS: Dict[str, ctypes.CDLL] = {}
_LIB_PATHS: Dict[str, str] = {}


class KernelTimer:
    """Times every kernel call of this module with a pair of events while it is active:

        with ops.KernelTimer() as timer: ...steps...
        timer.summary() -> {entry point: (calls, microseconds)}

    For measurement only: each call is bracketed on the current stream, so launches are not overlapped."""
    active: Optional["KernelTimer"] = None

    def __init__(self):
        self.records = []                 # (name, start event, end event)

    def __enter__(self):
        KernelTimer.active = self
        return self

    def __exit__(self, *exc):
        KernelTimer.active = None

    def call(self, name, fn, *args):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        out = fn(*args)
        b.record()
        self.records.append((name, a, b))
        return out

    def summary(self) -> Dict[str, Tuple[int, float]]:
        torch.cuda.synchronize()
        out: Dict[str, Tuple[int, float]] = {}
        for name, a, b in self.records:
            calls, us = out.get(name, (0, 0.0))
            out[name] = (calls + 1, us + a.elapsed_time(b) * 1e3)
        return out


class _Timed:
    """A kernel library whose entry points that launch something report to the active `KernelTimer`, if there is one."""
    __slots__ = ("_lib", "_short")

    def __init__(self, lib: ctypes.CDLL):
        object.__setattr__(self, "_lib", lib)
        object.__setattr__(self, "_short", {})

    def __getattr__(self, name):
        fn = getattr(self._lib, name)
        if KernelTimer.active is None or name not in _LAUNCHING:
            return fn
        timer = KernelTimer.active
        return lambda *args: timer.call(name[3:], fn, *args)


_C_TYPES = {"int": ctypes.c_int, "long long": ctypes.c_longlong, "unsigned long long": ctypes.c_ulonglong,
            "float": ctypes.c_float, "double": ctypes.c_double, "hipStream_t": ctypes.c_void_p, "size_t": ctypes.c_size_t}
_DECLARATIONS: Dict[str, Tuple[object, list]] = {}
_LAUNCHING: set = set()                                     # the entry points that take a stream: the others are questions to the host


def _declarations() -> Dict[str, Tuple[object, list]]:
    """Entry point -> (result type, argument types), read from the header that declares them (`csrc/api.h`): with the
    types known, ctypes converts plain integers to pointers itself, and a call's arguments need no objects around them
    (0.3 us each, a thousand a step)."""
    if _DECLARATIONS:
        return _DECLARATIONS
    import re
    with open(os.path.join(_build.CSRC, "api.h")) as f:
        text = re.sub(r"//[^\n]*", "", f.read())

    def ctype(decl: str):
        decl = decl.strip()
        if "*" in decl:
            return ctypes.c_char_p if decl.replace("const", "").replace("*", "").split()[0] == "char" else ctypes.c_void_p
        words = [w for w in decl.replace("const", "").split()]
        for n in (3, 2, 1):                                 # the type's words, with or without a parameter's name behind them
            for cut in (words[:n],):
                if " ".join(cut) in _C_TYPES and len(words) - n <= 1:
                    return _C_TYPES[" ".join(cut)]
        raise KernelError(f"api.h: no ctypes type for {decl!r}")

    for m in re.finditer(r"\b(int|long long|void|const char\s*\*)\s+(ia_\w+)\s*\(([^)]*)\)\s*;", text):
        result, name, params = m.group(1), m.group(2), m.group(3).strip()
        args = [] if params in ("", "void") else [ctype(a) for a in params.split(",")]
        restype = None if result == "void" else (ctypes.c_char_p if "char" in result else _C_TYPES[result])
        _DECLARATIONS[name] = (restype, args)
        if "hipStream_t" in params:
            _LAUNCHING.add(name)
    for must in ("ia_last_error", "ia_add_rmsnorm", "ia_gemm_skinny_bf16", "ia_attention_mfma", "ia_sample"):
        if must not in _DECLARATIONS:
            _DECLARATIONS.clear()
            raise KernelError(f"api.h: the declaration of {must} was not found (the header's form has changed?)")
    return _DECLARATIONS


def _declare(lib: ctypes.CDLL) -> None:
    for name, (restype, args) in _declarations().items():
        try:
            fn = getattr(lib, name)
        except AttributeError:                              # (an entry point of another library)
            continue
        fn.restype, fn.argtypes = restype, args


def library(target: str = "core"):
    """A compiled kernel library; compiled on first use when no built one is found."""
    lib = _LIBS.get(target)
    if lib is not None:
        return lib if KernelTimer.active is None else _Timed(lib)
    path = _build.library_path(target)
    if path is None:
        path = _build.build(target, verbose=True)
    lib = ctypes.CDLL(path)
    lib.ia_last_error.restype = ctypes.c_char_p
    if lib.ia_abi_version() != 1:
        raise KernelError(f"{path}: unexpected ABI version {lib.ia_abi_version()}")
    _declare(lib)
    _LIBS[target], _LIB_PATHS[target] = lib, path
    return lib if KernelTimer.active is None else _Timed(lib)


def _raw_library(target: str = "core") -> ctypes.CDLL:
    """The library without the timer around its entry points (for calls that a caller times under a name of its own)."""
    library(target)
    return _LIBS[target]


def library_files() -> Dict[str, str]:
    """The libraries loaded so far: target -> file."""
    return dict(_LIB_PATHS)


def require_gpu() -> None:
    if not torch.cuda.is_available():
        raise KernelError("inferrs_amd runs on an AMD GPU through its HIP kernels; "
                          "no GPU is visible and there is no CPU fallback")
    library()


def _check(code: int, target: str = "core") -> None:
    if code:
        raise KernelError(library(target).ia_last_error().decode("utf-8", "replace"))


def _stream() -> int:
    # (the raw handle straight from the runtime: `torch.cuda.current_stream()` builds a Python object around it, 3 us
    # a kernel call)
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _p(t: Optional[torch.Tensor]) -> Optional[int]:
    """A tensor's address as the entry points take it (their argument types are declared: see `_declarations`)."""
    return None if t is None else t.data_ptr()


def _dt(t: torch.Tensor) -> int:
    try:
        return _DT[t.dtype]
    except KeyError:
        raise KernelError(f"kernels take float32 or bfloat16 tensors, got {t.dtype}") from None


def _dev(*ts: Optional[torch.Tensor]) -> None:
    for t in ts:
        if t is not None and (not t.is_cuda or not t.is_contiguous()):
            raise KernelError("kernel operands must be contiguous GPU tensors "
                              f"(got device={t.device}, contiguous={t.is_contiguous()}, shape={tuple(t.shape)})")


def _i32(t: torch.Tensor, name: str) -> None:
    if t.dtype != torch.int32:
        raise KernelError(f"{name} must be int32, got {t.dtype}")


def _f32(t: Optional[torch.Tensor], name: str) -> None:
    if t is not None and t.dtype != torch.float32:
        raise KernelError(f"{name} must be float32, got {t.dtype}")


# ---- embedding, gathers ---------------------------------------------------------------------

def embed_gather(table: torch.Tensor, ids: torch.Tensor) -> torch.Tensor:
    _dev(table, ids); _i32(ids, "ids")
    vocab, hidden = table.shape
    n = ids.numel()
    out = torch.empty((n, hidden), dtype=table.dtype, device=table.device)
    _check(library().ia_embed_gather(_p(out), _p(table), _p(ids), n, hidden, vocab, _dt(table), _stream()))
    return out


def gather_rows(x: torch.Tensor, rows: torch.Tensor) -> torch.Tensor:
    _dev(x, rows); _i32(rows, "rows")
    n, cols = rows.numel(), x.shape[-1]
    out = torch.empty((n, cols), dtype=x.dtype, device=x.device)
    _check(library().ia_gather_rows(_p(out), _p(x), _p(rows), n, cols, _dt(x), _stream()))
    return out


# ---- norms ----------------------------------------------------------------------------------

def rmsnorm(x: torch.Tensor, w: torch.Tensor, eps: float, add_one: bool = False) -> torch.Tensor:
    _dev(x, w); _f32(w, "norm weight")
    cols = x.shape[-1]
    if w.numel() != cols:
        raise KernelError(f"rmsnorm: weight has {w.numel()} entries, rows have {cols}")
    rows = x.numel() // cols
    out = torch.empty_like(x)
    _check(library().ia_rmsnorm(_p(out), _p(x), _p(w), ctypes.c_float(eps), rows, cols, int(add_one),
                                _dt(x), _stream()))
    return out


def add_rmsnorm(x: torch.Tensor, delta: torch.Tensor, w: torch.Tensor, eps: float,
                add_one: bool = False) -> torch.Tensor:
    """x += delta in place (summed in 32-bit); returns rmsnorm(x)."""
    _dev(x, delta, w); _f32(w, "norm weight")
    if x.shape != delta.shape or x.dtype != delta.dtype:
        raise KernelError(f"add_rmsnorm: x {tuple(x.shape)} {x.dtype} and delta {tuple(delta.shape)} {delta.dtype} differ")
    cols = x.shape[-1]
    if w.numel() != cols:
        raise KernelError(f"add_rmsnorm: weight has {w.numel()} entries, rows have {cols}")
    rows = x.numel() // cols
    out = torch.empty_like(x)
    _check(library().ia_add_rmsnorm(_p(out), _p(x), _p(delta), _p(w), ctypes.c_float(eps), rows, cols,
                                    int(add_one), _dt(x), _stream()))
    return out


def add_inplace(x: torch.Tensor, delta: torch.Tensor) -> torch.Tensor:
    _dev(x, delta)
    if x.shape != delta.shape or x.dtype != delta.dtype:
        raise KernelError("add_inplace: operands differ in shape or dtype")
    _check(library().ia_add_inplace(_p(x), _p(delta), ctypes.c_longlong(x.numel()), _dt(x), _stream()))
    return x


# The activations a gated feed-forward may name, and their numbers in the kernels' `dual` / `act` argument
# (0 there: a plain product).  "gelu_tanh" is GELU in its tanh form, x / 2 * (1 + tanh(sqrt(2 / pi) * (x + 0.044715 x^3))).
ACTIVATIONS: Dict[str, int] = {"silu": 1, "gelu_tanh": 2}


def activation_code(activation: str) -> int:
    try:
        return ACTIVATIONS[activation]
    except KeyError:
        raise KernelError(f"no kernel has the activation {activation!r}; known: {sorted(ACTIVATIONS)}") from None


def gate_mul(gu: torch.Tensor, activation: str = "silu") -> torch.Tensor:
    """rows of [gate | up] -> act(gate) * up."""
    _dev(gu)
    if gu.shape[-1] % 2:
        raise KernelError(f"gate_mul: last dimension {gu.shape[-1]} must be even")
    inter = gu.shape[-1] // 2
    rows = gu.numel() // (2 * inter)
    out = torch.empty((*gu.shape[:-1], inter), dtype=gu.dtype, device=gu.device)
    _check(library().ia_gate_mul(_p(out), _p(gu), rows, inter, activation_code(activation), _dt(gu), _stream()))
    return out


def silu_mul(gu: torch.Tensor) -> torch.Tensor:
    """rows of [gate | up] -> silu(gate) * up."""
    return gate_mul(gu, "silu")


def add_bias(x: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    """x[row] += bias in place, for products whose kernel has no place for a bias."""
    _dev(x, bias)
    cols = x.shape[-1]
    if bias.numel() != cols or bias.dtype != x.dtype:
        raise KernelError(f"add_bias: a bias of {bias.numel()} {bias.dtype} entries for rows of {cols} {x.dtype}")
    _check(library().ia_add_bias(_p(x), _p(bias), x.numel() // cols, cols, _dt(x), _stream()))
    return x


# ---- position encoding ----------------------------------------------------------------------

def rope_table(positions: torch.Tensor, inv_freq: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    _dev(positions, inv_freq); _i32(positions, "positions"); _f32(inv_freq, "inv_freq")
    n, half = positions.numel(), inv_freq.numel()
    cos = torch.empty((n, half), dtype=torch.float32, device=positions.device)
    sin = torch.empty_like(cos)
    _check(library().ia_rope_table(_p(cos), _p(sin), _p(positions), _p(inv_freq), n, half, _stream()))
    return cos, sin


def qk_rope_kv(qkv: torch.Tensor, nq: int, nkv: int, d: int, *,
               q_norm_w: Optional[torch.Tensor], k_norm_w: Optional[torch.Tensor],
               eps: float, add_one: bool, cos: Optional[torch.Tensor], sin: Optional[torch.Tensor],
               rot: int, interleaved: bool, k_cache: Optional[torch.Tensor],
               v_cache: Optional[torch.Tensor], slots: Optional[torch.Tensor],
               page_size: int) -> torch.Tensor:
    """Norm and rotate q and k, write k and v at `slots` of the cache; returns q [n, nq, d].  `qkv` may be a product still split
    along its k (`Partials`), where the step's sizes are taken that way and there is a rotation and a cache to write."""
    parts = None
    if isinstance(qkv, Partials):
        splits, n, width = qkv.parts.shape
        # (that kernel reads everything in 16-byte pieces; arrays that begin elsewhere go with the stored product)
        arrays = (q_norm_w, k_norm_w, cos, sin, k_cache, v_cache, qkv.parts)
        if (cos is None or slots is None or k_cache is None or k_cache.dtype != torch.bfloat16 or width != (nq + 2 * nkv) * d
                or not qk_rope_kv_partials_fits(n, d, rot, interleaved, page_size)
                or any(t is not None and t.data_ptr() % 16 for t in arrays)):
            qkv = qkv.materialize()
        else:
            parts, qkv = qkv.parts, qkv.parts[0]
    _dev(qkv, q_norm_w, k_norm_w, cos, sin, k_cache, v_cache, slots)
    _f32(q_norm_w, "q_norm weight"); _f32(k_norm_w, "k_norm weight"); _f32(cos, "cos"); _f32(sin, "sin")
    n = qkv.shape[0]
    if qkv.dim() != 2 or qkv.shape[1] != (nq + 2 * nkv) * d:
        raise KernelError(f"qk_rope_kv: qkv has shape {tuple(qkv.shape)}, expected [n, {(nq + 2 * nkv) * d}]")
    for w, name in ((q_norm_w, "q_norm"), (k_norm_w, "k_norm")):
        if w is not None and w.numel() != d:
            raise KernelError(f"qk_rope_kv: {name} weight has {w.numel()} entries, head_dim is {d}")
    if cos is not None:
        if sin is None or cos.shape != (n, rot // 2) or sin.shape != cos.shape:
            raise KernelError(f"qk_rope_kv: rotary tables must be [{n}, {rot // 2}]")
    if slots is not None:
        _i32(slots, "slots")
        if k_cache is None or v_cache is None:
            raise KernelError("qk_rope_kv: slots given without a cache")
        if slots.numel() != n:
            raise KernelError(f"qk_rope_kv: {slots.numel()} slots for {n} tokens")
        _check_cache(k_cache, v_cache, nkv, page_size, d, qkv.dtype if parts is None else torch.bfloat16, "qk_rope_kv")
    q_out = torch.empty((n, nq, d), dtype=qkv.dtype if parts is None else torch.bfloat16, device=qkv.device)
    if parts is not None:
        _check(library().ia_qk_rope_kv_partials(
            _p(q_out), _p(k_cache), _p(v_cache), _p(parts), parts.shape[0], _p(q_norm_w), _p(k_norm_w), _p(cos), _p(sin), _p(slots),
            n, nq, nkv, d, page_size, ctypes.c_float(eps), int(add_one), _stream()))
        return q_out
    _check(library().ia_qk_rope_kv(
        _p(q_out), _p(k_cache if slots is not None else None), _p(v_cache if slots is not None else None),
        _p(qkv), _p(q_norm_w), _p(k_norm_w), _p(cos), _p(sin), _p(slots), n, nq, nkv, d, rot,
        int(interleaved), page_size, ctypes.c_float(eps), int(add_one), _dt(qkv), _stream()))
    return q_out


@functools.lru_cache(maxsize=4096)
def qk_rope_kv_partials_fits(n: int, d: int, rot: int, interleaved: bool, page_size: int) -> bool:
    """Whether `qk_rope_kv` reads projections that are still split along their k (`Partials`) in a step of `n` tokens."""
    return bool(library().ia_qk_rope_kv_partials_fits(n, d, rot, int(interleaved), page_size))


def qk_rope_kv_strided(proj: torch.Tensor, nq: int, nkv: int, d: int, dv: int, *, q_off: int, k_off: Optional[int],
                       v_off: Optional[int], q_norm_w: Optional[torch.Tensor], k_norm_w: Optional[torch.Tensor], eps: float,
                       add_one: bool, cos: Optional[torch.Tensor], sin: Optional[torch.Tensor], rot: int, interleaved: bool,
                       k_cache: Optional[torch.Tensor], v_cache: Optional[torch.Tensor], slots: Optional[torch.Tensor],
                       page_size: int, v_with: Optional[torch.Tensor] = None, v_mix: float = 0.0) -> torch.Tensor:
    """`qk_rope_kv` on rows of any layout: a row of `proj` holds the query heads from `q_off`, the key heads from `k_off`
    and the value heads (`dv` wide each) from `v_off`, and whatever else beside them.  `k_off` None: the rows hold no keys
    or values (a layer that reads another layer's cache).  `v_with` [n, nkv * dv] (rows any distance apart): another layer's
    values of the same tokens; (1 - v_mix) v + v_mix v_with is what is cached.  Returns q [n, nq, d]."""
    _dev(proj, q_norm_w, k_norm_w, cos, sin, k_cache, v_cache, slots)
    if v_with is not None and (not v_with.is_cuda or tuple(v_with.shape) != (proj.shape[0], nkv * dv) or v_with.dtype != proj.dtype
                               or v_with.stride(1) != 1):
        raise KernelError(f"qk_rope_kv_strided: values to mix with {tuple(v_with.shape)} {v_with.dtype} are no {nkv} heads of {dv}")
    _f32(q_norm_w, "q_norm weight"); _f32(k_norm_w, "k_norm weight"); _f32(cos, "cos"); _f32(sin, "sin")
    if proj.dim() != 2 or proj.stride(1) != 1:
        raise KernelError(f"qk_rope_kv_strided: the projections are 2-D rows, got {tuple(proj.shape)}")
    n, ld_ = proj.shape[0], proj.stride(0)
    for w, name in ((q_norm_w, "q_norm"), (k_norm_w, "k_norm")):
        if w is not None and w.numel() != d:
            raise KernelError(f"qk_rope_kv_strided: {name} weight has {w.numel()} entries, head_dim is {d}")
    if cos is not None and (sin is None or cos.shape != (n, rot // 2) or sin.shape != cos.shape):
        raise KernelError(f"qk_rope_kv_strided: rotary tables must be [{n}, {rot // 2}]")
    if q_off < 0 or q_off + nq * d > proj.shape[1]:
        raise KernelError(f"qk_rope_kv_strided: {nq} query heads of {d} at {q_off} do not fit rows of {proj.shape[1]}")
    if k_off is None:
        slots = None
    if slots is not None:
        _i32(slots, "slots")
        if k_cache is None or v_cache is None or v_off is None or slots.numel() != n:
            raise KernelError("qk_rope_kv_strided: slots need a cache, the values' place and one entry a token")
        if k_off < 0 or v_off < 0 or k_off + nkv * d > proj.shape[1] or v_off + nkv * dv > proj.shape[1]:
            raise KernelError(f"qk_rope_kv_strided: keys at {k_off} / values at {v_off} do not fit rows of {proj.shape[1]}")
        _check_cache(k_cache, v_cache, nkv, page_size, d, proj.dtype, "qk_rope_kv_strided", dv)
    q_out = torch.empty((n, nq, d), dtype=proj.dtype, device=proj.device)
    _check(library().ia_qk_rope_kv_strided(
        _p(q_out), _p(k_cache if slots is not None else None), _p(v_cache if slots is not None else None), _p(proj),
        _p(q_norm_w), _p(k_norm_w), _p(cos), _p(sin), _p(slots), n, ld_, q_off, -1 if k_off is None else k_off,
        -1 if v_off is None else v_off, nq, nkv, d, dv, rot, int(interleaved), page_size, ctypes.c_float(eps), int(add_one),
        _p(v_with), v_with.stride(0) if v_with is not None else 0, ctypes.c_float(v_mix), _dt(proj), _stream()))
    return q_out


# ---- attention --------------------------------------------------------------------------------

def _check_cache(k_cache: torch.Tensor, v_cache: torch.Tensor, nkv: int, page_size: int, d: int,
                 dtype: torch.dtype, who: str, dv: Optional[int] = None) -> None:
    """Keys [pages, nkv, page_size, d]; values transposed inside a page, [pages, nkv, dv, page_size] (dv None: d)."""
    dv = d if dv is None else dv
    if (k_cache.dtype != dtype or v_cache.dtype != dtype or k_cache.dim() != 4 or v_cache.dim() != 4
            or tuple(k_cache.shape[1:]) != (nkv, page_size, d) or tuple(v_cache.shape[1:]) != (nkv, dv, page_size)
            or k_cache.shape[0] != v_cache.shape[0]):
        raise KernelError(f"{who}: cache has shapes {tuple(k_cache.shape)} {k_cache.dtype} and "
                          f"{tuple(v_cache.shape)} {v_cache.dtype}, expected [pages, {nkv}, {page_size}, {d}] "
                          f"and [pages, {nkv}, {dv}, {page_size}] {dtype}")


PORTIONS_ROUND = 340           # tiles of 64 keys that the matrix cores' blocks have under way together (two blocks a compute unit)
PORTIONS_PLAIN_ROUND = 1200    # and the plain kernel's waves
PORTIONS_TILE = 64             # keys of a tile, and columns (token, query head of a key/value head) of a block


def attention_portions_pay(q_lens: Sequence[int], kv_starts: Sequence[int], nq: int, nkv: int, d: int,
                           span: Optional[int] = None) -> bool:
    """Whether 32-bit portions of prompts (`q_lens` tokens behind `kv_starts` cached ones, in the step's order) are faster on the
    matrix cores (`attention_generic(portions=True)`) than with the plain kernel.  There, a block of 64 columns walks the contexts of
    its requests one after the other, mostly with idle columns where portions are short; here a wave walks each token's.  A block's
    chains start with the longest, so that they take the longer of the longest chain of tiles and of all tiles over what the chip has
    under way; the plain kernel, whose longest may start late, half of the shorter of the two besides.  A tile of the plain kernel's
    chain takes 0.97, 1.1, 1.2 and 1.35 (one to four heads a wave, head size 64: 6.3 to 9.2 us against 6.5) and 1.12, 1.25, 1.4 and 1.5
    times (128: 10.5 to 14.2 against 9.4) that of a block's; `tile` asks for some fifteen parts in a hundred more.  `span`: a window's
    or a chunk's positions.
    Measured over 2,219 steps (1 to 128 requests of 2 to 1,200 tokens, alike, of all sizes, or few long ones beside short ones, contexts
    up to 8,000, windows, some thirty pairs of head counts): the time of the faster kernel is 0.985 of the chosen one's in the mean, 15
    steps lose more than 5 % against the plain kernel (the worst 0.71 of its speed, 139 us).  Asking for eight tokens a request in the
    mean, as an earlier rule did: 0.947, 266 steps, the worst 0.06 (16/8 heads of 128, 64 requests of 2 tokens at 4,000 beside one of 500
    1,513 us by the plain kernel, 9,095 on the matrix cores; 16 requests of 8 at 500 156 and 281)."""
    g = nq // nkv
    heads, groups = min(g, 4), -(-g // 4)
    chain = plain_chain = total = plain_total = 0
    block, here, col = -1, 0, 0                             # the last request's last block, and the tiles of that block so far
    for q, start in zip(q_lens, kv_starts):
        tiles = plain = (start + q - 1) // PORTIONS_TILE + 1
        if span:
            plain = min(tiles, span // PORTIONS_TILE + 2)
            tiles = min(tiles, (span + min(q, -(-PORTIONS_TILE // g))) // PORTIONS_TILE + 2)
        first, last = col // PORTIONS_TILE, (col + q * g - 1) // PORTIONS_TILE
        here = here + tiles if first == block else tiles
        chain = max(chain, here)
        if last > first:
            here = tiles
        block = last
        col += q * g
        total += (last - first + 1) * tiles
        plain_chain = max(plain_chain, plain)
        plain_total += q * plain
    tile = (0.72 if d == 64 else 0.855) + 0.11 * heads
    load = plain_total * nkv * groups / PORTIONS_PLAIN_ROUND
    return max(chain, total * nkv / PORTIONS_ROUND) <= tile * (max(plain_chain, load) + 0.5 * min(plain_chain, load))


def attention_generic(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                      positions: torch.Tensor, token_seq: torch.Tensor, block_table: torch.Tensor,
                      *, window: Optional[int], scale: float, max_kv_len: Optional[int] = None,
                      split: Optional[bool] = None, sink: bool = False, mask_chunk: Optional[int] = None,
                      sinks: Optional[torch.Tensor] = None, keep_first: int = 0,
                      softcap: Optional[float] = None, portions: bool = False) -> torch.Tensor:
    """q [n, nq, d] against the paged cache (values may have a width of their own: v_cache [pages, nkv, dv, page_size],
    the result is [n, nq, dv]); token i sees the keys at positions <= positions[i]
    (and > positions[i] - window) of row token_seq[i] of the table.  Any head size up to 512, any
    page size, 32-bit or bfloat16 storage, all arithmetic in 32-bit.  `max_kv_len`: an upper bound of
    positions + 1 (default: what the table can hold).  Steps of few tokens run a wave a segment of 512 keys
    and a merge kernel (`split`; None: the kernel's own rule); the bits are the same either way.
    `sink`: the softmax's denominator holds one more term, exp(0): a key of score 0 that has no value; `sinks` [nq]
    (32-bit): the term is exp(sinks[h]) for query head h instead (not scaled).  `mask_chunk`: a token sees the keys of its
    own chunk of that many positions only (chunks counted from position 0 of the sequence), up to itself.  `keep_first`: it
    sees the first so many positions besides.  `softcap`: a score becomes softcap * tanh(score / softcap).  `portions`: the tokens
    are portions of prompts, several neighbours of each request, which 32-bit heads of 64 and 128 take on the matrix cores (the
    same bits; whether they are faster there is for `attention_portions_pay` to say)."""
    _dev(q, k_cache, v_cache, positions, token_seq, block_table, sinks)
    sink = _check_sinks(sinks, sink, q.shape[1])
    _i32(positions, "positions"); _i32(token_seq, "token_seq"); _i32(block_table, "block_table")
    n, nq, d = q.shape
    nkv, page_size = k_cache.shape[1], k_cache.shape[2]
    dv = v_cache.shape[2] if v_cache.dim() == 4 else d
    _check_cache(k_cache, v_cache, nkv, page_size, d, q.dtype, "attention", dv)
    if positions.numel() != n or token_seq.numel() != n or block_table.dim() != 2:
        raise KernelError("attention: positions, token_seq and block_table do not fit the batch")
    capacity = block_table.shape[1] * page_size
    max_kv_len = capacity if max_kv_len is None else min(int(max_kv_len), capacity)
    out = torch.empty((n, nq, dv), dtype=q.dtype, device=q.device)
    lib = library()
    if (portions and not split and q.dtype == torch.float32 and (out.data_ptr() | k_cache.data_ptr() | v_cache.data_ptr()) % 16 == 0
            and lib.ia_attention_portions_f32_fits(n, nq, nkv, d, dv, page_size, max_kv_len)):
        _check(lib.ia_attention_portions_f32(
            _p(out), _p(q), _p(k_cache), _p(v_cache), _p(positions), _p(token_seq), _p(block_table), n, block_table.shape[1], nq, nkv, d,
            page_size, int(window or 0), ctypes.c_float(scale), max_kv_len, int(bool(sink)), int(mask_chunk or 0), _p(sinks),
            int(keep_first), ctypes.c_float(softcap or 0.0), _stream()))
        return out
    ws_floats = lib.ia_attention_generic_workspace(n, nq, nkv, d, dv, max_kv_len) if split is not False else 0
    if split and not ws_floats:
        raise KernelError("attention: a step of this many tokens, or of so few keys, is not split")
    ws = torch.empty((ws_floats,), dtype=torch.float32, device=q.device) if ws_floats else None
    _check(lib.ia_attention_generic(
        _p(out), _p(q), _p(k_cache), _p(v_cache), _p(positions), _p(token_seq), _p(block_table), n,
        block_table.shape[1], nq, nkv, d, dv, page_size, int(window or 0), ctypes.c_float(scale), _dt(q),
        _p(ws), max_kv_len, int(bool(sink)), int(mask_chunk or 0), _p(sinks), int(keep_first), ctypes.c_float(softcap or 0.0),
        _stream()))
    return out


def _check_sinks(sinks: Optional[torch.Tensor], sink: bool, nq: int) -> bool:
    if sinks is None:
        return bool(sink)
    _f32(sinks, "sinks")
    if sinks.numel() != nq or not sinks.is_contiguous():
        raise KernelError(f"attention: {sinks.numel()} sink values for {nq} query heads")
    return True


ATTN_TARGET_WAVES = 2048       # waves wanted in flight before the keys stop being split
ATTN_MIN_CHUNK = 64            # fewest keys a split is worth


def attention_mfma_fits(dtype: torch.dtype, d: int, page_size: int, dv: Optional[int] = None) -> bool:
    """`dv`: the values' width where it is not the keys'."""
    return (dtype == torch.bfloat16 and d in _build.ATTN_HEAD_DIMS and page_size % 16 == 0
            and (dv is None or dv in _build.ATTN_HEAD_DIMS))


ATTN_TILE_COLS = 128           # head size 128, prompt portions: columns a block of four waves
ATTN_TILE_BLOCKS = 256         # compute units: a block's eight waves fill one
ATTN_TILE_MIN_CHUNK = 512      # fewest keys a block's share is worth (eight stages of 64)
ATTN_TILE_WHOLE_UP_TO = 2048   # contexts up to this length are not split
ATTN_TILE_FEW_UP_TO = 512     # fewer columns than a block has: keys that one walk takes whole


def attention_few_columns(n_seqs: int, nkv: int, g: int, max_q_len: int, d: int) -> bool:
    """Whether portions of so many tokens have fewer columns than a block of the kernel that shares keys between its waves, and run
    there in one round of blocks where their contexts are short."""
    return d == 128 and 16 < max_q_len * g < ATTN_TILE_COLS and n_seqs * nkv * -(-max_q_len * g // 64) <= ATTN_TILE_BLOCKS


def attention_split(n_seqs: int, nkv: int, g: int, max_q_len: int, max_kv_len: int, d: int = 0) -> Tuple[int, int]:
    """(splits, keys per split) for the matrix-core kernel: the keys are split between waves
    when the batch alone has too few (request, kv head, column block) items to fill the chip."""
    cols = max_q_len * g
    if d == 128 and cols >= ATTN_TILE_COLS:
        if 2 * max_q_len > max_kv_len or max_kv_len <= ATTN_TILE_WHOLE_UP_TO:
            # whole prompts and portions that span most of their context: a block's walk ends at its own tokens, so
            # the later splits of the early blocks are empty and the partial sums of every row go through memory for
            # nothing (16 query and 8 key/value heads, 1,024 tokens, 128 blocks: 25.6 us whole against 28.2 in two
            # splits; 2,048 tokens 44 against 63; 32 query heads, 512 tokens 18 against 26); short contexts likewise: the
            # walks are short, and where the blocks are few the kernel halves them instead (a portion of 512 tokens at
            # a context of 2,048, 32 query heads: 29.7 us whole in blocks of 64 columns against 36.8 in two splits)
            return 1, -(-max_kv_len // 64) * 64
        # In microseconds: whole, a key takes a block of 64 columns (which the kernel takes for few blocks that are not split)
        # 0.0119 and one of 128 0.0172 a round of the compute units; in shares 0.0175, and a round's worth of partial sums 10.3 to
        # write, read and merge; 2.5 % from the measurements in the mean.  Whole against 2, 3 and 4 shares, 40 query heads: 512 tokens
        # at 6,000 keys 113, 128, 99 and 115, at 16,384 293, 304, 221 and 246; 1,024 tokens at 3,000 keys 98, 117, 117 and 128 (their
        # early blocks walk less than the context: `max_q_len` / 2); 32 query heads, 256 tokens at 4,096 57, 56, 74 and 64; five query heads a
        # key head, 32 tokens at 2,304 34, 32, 26 and 25.  Against powers of two up to one block a compute unit: 1.16 times as fast
        # in the mean of 142 sizes at which the two differ, 0.95 (1.6 us) to 1.49.
        items = n_seqs * nkv * -(-cols // ATTN_TILE_COLS)
        if 2 * items <= ATTN_TILE_BLOCKS:
            best = 6.0 + 0.0119 * max_kv_len
        else:
            best = 15.0 + 0.0172 * (max_kv_len - max_q_len // 2) * -(-items // ATTN_TILE_BLOCKS)
        splits = 1
        for ways in range(2, 129):
            chunk = -(-(-(-max_kv_len // ways)) // 64) * 64
            if chunk < ATTN_TILE_MIN_CHUNK:
                break
            cost = 10.2 + 0.18 * ways + 10.3 * items * ways / ATTN_TILE_BLOCKS + 0.0175 * chunk * -(-items * ways // ATTN_TILE_BLOCKS)
            if cost < best:
                best, splits = cost, ways
        chunk = -(-max_kv_len // splits)
        return splits, -(-chunk // 64) * 64
    if max_kv_len <= ATTN_TILE_FEW_UP_TO and attention_few_columns(n_seqs, nkv, g, max_q_len, d):
        # few columns in one round of blocks that share their keys: whole (40 tokens behind 100, two query heads a key head, 12.8 us
        # in two splits of single waves, 7.6 whole; 20 tokens behind 450 12.1 in four, 10.5 whole; 177 sizes 1.06 to 2.39 times as fast)
        return 1, -(-max_kv_len // 64) * 64
    col_blocks = 1 if cols <= 16 else -(-cols // 32)
    items = n_seqs * nkv * col_blocks
    splits = 1
    while items * splits < ATTN_TARGET_WAVES and max_kv_len >= 2 * splits * ATTN_MIN_CHUNK and splits < 128:
        splits *= 2
    chunk = -(-max_kv_len // splits)
    chunk = -(-chunk // 32) * 32
    return splits, chunk


DECODE_WAVES = 1024            # as many waves as the chip has SIMDs (head sizes up to 128 have room for two on each, see below)
DECODE_MIN_CHUNK = 64          # fewest keys a wave's share is worth (two steps of 32); 128 up to a context of 512
DECODE_MANY_SPLITS = 32        # more splits than these only where a split would still hold more than 128 keys


def decode_split(n_seqs: int, nkv: int, g: int, max_kv_len: int) -> Tuple[int, int]:
    """(splits, keys per split) for the decode kernel: the largest power of two that keeps the step's waves
    (request x kv head x 16 query heads x split) within one round of the chip and a wave's share at 64 keys
    or more; beyond 32 splits (eight blocks to merge) only where a share would exceed 128 keys.  Measured at head
    size 128, 32 query and 8 kv heads, context 8,192 (microseconds a layer): batch 1
    17.8 with 64 splits against 21.3 with 32, batch 4 31.3 with 32 against 36.7 with 16.  A SIMD has the registers for two waves up to a
    head size of 128, and twice the waves, two rounds' worth side by side, are slower up to 32 requests (batch 4 37.3, batch 8 56.2
    against 51.3 and at 2,000 18.4 against 17.4, batch 16 at 1,500 25.6 against 24.8, batch 32 at 1,500 43.2 against 37.8): more partial
    results to hand over, and one wave's loads keep a SIMD's share of the memory busy; at 64 requests they are 1 to 5 % faster (700 keys
    36.0 against 37.2, 1,500 71.1 and 72.0, 4,000 177.6 and 187.3): not taken.  Shares of 64 keys against 128:
    batch 1 at 2,048 9.3 against 11.8; batch 4 12.6 against 14.1; batch 8 17.6 against 21.1; and 64 splits of 64 keys at 4,096 lose
    to 32 of 128 (batch 2, an earlier kernel: 17.0 against 16.0).  Shares of 32 keys at a bound of 1,024 are worth 0.2 to 1.0 us to one
    to four requests (16 query heads, batch 1, 700 keys 8.0 against 8.7) and lose at eight (12.6 against 11.3): not taken."""
    items = n_seqs * nkv * -(-g // 16)
    min_chunk = DECODE_MIN_CHUNK if max_kv_len > 512 else 128
    splits = 1
    while items * splits * 2 <= DECODE_WAVES and max_kv_len >= 2 * splits * min_chunk and splits < 128:
        if splits >= DECODE_MANY_SPLITS and max_kv_len <= splits * 128:
            break
        splits *= 2
    chunk = -(-max_kv_len // splits)
    return splits, -(-chunk // 32) * 32


@functools.lru_cache(maxsize=4096)
def decode_shares(n_seqs: int, nkv: int, g: int, max_kv_len: int, d: int = 128, dv: int = 128) -> Tuple[int, int]:
    """(splits, keys per split) that a decode step takes: `decode_split`'s, but for other counts where they were faster, at keys of `d` and values
    of `dv` features.  Measured at widths of (64, 64), (128, 128), (128, 64), (192, 192) and (256, 256), 1 to 64 requests of 1 to 8 key heads with 1
    to 16 query heads, contexts within a bound's last bucket and of 40 to 97 % of it (8 to 97 % of 1,024); speed against `decode_split`'s counts,
    means at these widths in this order:
    - a round's worth of waves that eight splits leave idle goes to twelve: 1.11, 1.10, 1.16, 1.15, 1.17, none below 0.98;
    - up to 1,024 keys four splits meet in one block where eight are handed over between two: 1.11, 1.01, 1.03 (contexts up to 700 keys 1.13 to
      1.16, longer ones 0.88 to 1.07); 0.93 and 0.96 with wider heads, which keep eight;
    - 48 splits for 32 of 3,072 to 4,095 keys with up to eight query heads a key head: 1.04, 1.08, 1.11, 1.14; with sixteen 0.95 to 1.03, and 0.92 at
      256 (what a block hands over is as wide as its query heads are); 64 of 4,096 keys with up to four: 1.02, 1.07, 1.08, 1.14; with more 0.91 to
      0.98, and 0.86 at 256;
    - 28 splits for 32, which leave some of the chip's waves out: from 28 pairs of a request and a key head on at 8,192 keys and more 1.03, 1.08, 1.02, 1.05,
      1.00, with fewer 0.97, 1.00, 0.94, 0.96, 0.94; from 17 on at 3,072 to 4,095 keys 1.02, 1.06, 1.03, 1.04, at 256 0.87 to 1.19.
    (Blocks of three waves for four: 0.95, 1.00, 0.99, 1.00, 1.01, not taken.)"""
    splits, chunk = decode_split(n_seqs, nkv, g, max_kv_len)
    items = n_seqs * nkv * -(-g // 16)
    wide = max(d, dv)
    other = splits
    if splits == 8 and 512 < max_kv_len <= 1024:
        if wide <= 128:
            other = 4
    elif splits == 8 and items * 12 <= DECODE_WAVES and max_kv_len >= 2048:
        other = 12
    elif splits == 32 and wide < 256 and 3072 <= max_kv_len < 4096 and items > 16:
        other = 28
    elif splits == 32 and wide < 256 and 3072 <= max_kv_len < 4096 and g <= 8:
        other = 48
    elif splits == 32 and wide < 256 and max_kv_len == 4096 and items <= 16 and g <= 4:
        other = 64
    elif splits == 32 and items >= 28 and max_kv_len >= 8192:
        other = 28
    if other == splits:
        return splits, chunk
    return other, -(-(-(-max_kv_len // other)) // 32) * 32


@functools.lru_cache(maxsize=4096)
def decode_fused_pays(n_seqs: int, nkv: int, g: int, d: int, dv: int, max_kv_len: int, span: int, *, formed: bool, gated: bool) -> bool:
    """Whether `attention_decode_fused` is faster than the kernels that it stands for: the norm and rotation, `attention_mfma` with its merge and (`gated`)
    the gate; or, of queries that are `formed` already, the attention and its merge alone.  `span`: the keys that a token sees at most
    (a window, a chunk of the mask; 0: all).  What the decode kernel pays for one launch is the hand-over: the last block of a (request, key head)
    reads all others' partial results past the caches, which the merge's kernel spreads over the chip; and where keys and values are wide, a
    wave's registers.  Measured at the widths of `decode_shares` and at 700 drawn sizes, (64, 256) among them: 1 to 73 requests of 1 to 8 key heads
    with 1 to 16 query heads, 512 to 16,384 keys, windows of 128 to 2,048 (times of the separate kernels over this one's, by the floats that one merge
    reads; a pair is a request and a key head).  Over all of these sizes the choice is 0.2 to 2 % off the faster one in the mean:
    - layers, widths up to 128: 1.3 to 1.8 in the mean with nothing handed over, 1.2 to 1.5 below 8,192 floats, 1.1 to 1.3 at 8,192; at 16,384 1.07 to
      1.16 with a gate (fewer than eight pairs 0.87 to 1.16) and 0.94 to 1.01 without, beyond that 0.5 to 0.95.  Without a gate, where a share is
      as long as a window of 1,024 and more, two waves of a pair have work: up to 127 pairs 0.94 in the mean;
    - up to 384 features of a key and a value, up to eight query heads a key head: 1.1 to 1.5 up to 4,096 floats, 1.0 to 1.15 with a gate and 0.9 to 1.03
      without up to 8,192, 0.6 to 1.0 beyond; with more query heads 0.4 to 1.8, 0.7 in the mean.  (256, 256): 0.17 to 1.16, but 1.06 to 1.6 from
      192 pairs on in one block under windows and up to 1,024 keys;
    - formed queries: from 64 pairs on 1.2 in the mean, and for 64 features in one block, else 0.86 (0.74 at (64, 256) and (192, 192)).  Under windows
      shorter than a quarter of the bound from an eighth of the window on: 32 pairs and a window of 128 1.29, 64 and 512 1.02, 128 and 1,024 1.12, 64
      and 1,024 0.87."""
    splits, chunk = decode_shares(n_seqs, nkv, g, max_kv_len, d, dv)
    nq = nkv * g
    blocks = _decode_sizes(_build.attn_target(d, dv), 1, nq, nkv, splits)[0] // (nq * (dv + 2)) or 1
    handed = min(g, 16) * dv * blocks if blocks > 1 else 0
    items = n_seqs * nkv * -(-g // 16)
    narrow = 0 < 4 * span <= max_kv_len
    if d + dv > 384:
        return blocks == 1 and items >= 192 and (0 < span < max_kv_len or (max_kv_len <= 1024 and items <= 256))
    small = max(d, dv) <= 128
    if formed:
        if narrow:
            return items >= max(32 if small else 64, span // 8)
        return items >= 64 or (small and d <= 64 and blocks == 1)
    if not small:
        return g <= 8 and handed <= (8192 if gated else 4096)
    if not gated and narrow and 1024 <= span <= chunk and items < 128:
        return False
    return handed < 16384 or (gated and handed == 16384 and items >= 8)


def attention_mfma(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, positions: torch.Tensor,
                   cu_tokens: torch.Tensor, block_table: torch.Tensor, *, max_q_len: int, max_kv_len: int,
                   window: Optional[int], scale: float, splits: Optional[int] = None,
                   seqs: Optional[Tuple[int, int]] = None, tokens: Optional[Tuple[int, int]] = None,
                   out: Optional[torch.Tensor] = None, sink: bool = False, mask_chunk: Optional[int] = None,
                   sinks: Optional[torch.Tensor] = None, keep_first: int = 0, softcap: Optional[float] = None) -> torch.Tensor:
    """The matrix-core kernel: bfloat16, head sizes in steps of 16 up to 256, page sizes in steps
    of 16.  Request s owns tokens cu_tokens[s]..cu_tokens[s+1] at consecutive positions.  `seqs` =
    (first, count) and `tokens` = (first, count) restrict the call to a run of requests and their
    tokens (the whole step by default); `max_q_len` and `max_kv_len` are the largest token count of
    one of these requests in this step and their largest length after it.  `out` receives the result
    (rows outside `tokens` are left alone).  `sink`, `sinks`, `mask_chunk`, `keep_first`, `softcap`: as in
    `attention_generic`."""
    _dev(q, k_cache, v_cache, positions, cu_tokens, block_table, out, sinks)
    sink = _check_sinks(sinks, sink, q.shape[1])
    _i32(positions, "positions"); _i32(cu_tokens, "cu_tokens"); _i32(block_table, "block_table")
    n, nq, d = q.shape
    nkv, page_size = k_cache.shape[1], k_cache.shape[2]
    dv = v_cache.shape[2] if v_cache.dim() == 4 else d
    _check_cache(k_cache, v_cache, nkv, page_size, d, q.dtype, "attention", dv)
    if not attention_mfma_fits(q.dtype, d, page_size, dv):
        raise KernelError(f"attention_mfma: takes bfloat16, head sizes {_build.ATTN_HEAD_DIMS[0]}.."
                          f"{_build.ATTN_HEAD_DIMS[-1]} in steps of 16 and page sizes in steps of 16; got "
                          f"{q.dtype}, head size {d}, page size {page_size}")
    all_seqs = cu_tokens.numel() - 1
    seq_begin, n_seqs = seqs if seqs is not None else (0, all_seqs)
    token_begin, n_tokens = tokens if tokens is not None else (0, n)
    if (positions.numel() != n or block_table.dim() != 2 or block_table.shape[0] < all_seqs or nq % nkv
            or seq_begin < 0 or seq_begin + n_seqs > all_seqs or token_begin < 0 or token_begin + n_tokens > n):
        raise KernelError("attention_mfma: positions, cu_tokens, block_table and the ranges do not fit the batch")
    if max_kv_len > block_table.shape[1] * page_size or max_q_len < 1 or max_q_len > max(n_tokens, 1):
        raise KernelError(f"attention_mfma: max_kv_len {max_kv_len} / max_q_len {max_q_len} do not fit "
                          f"{block_table.shape[1]} pages of {page_size} and {n_tokens} tokens")
    if out is None:
        out = torch.empty((n, nq, dv), dtype=q.dtype, device=q.device)
    elif tuple(out.shape) != (n, nq, dv) or out.dtype != q.dtype:
        raise KernelError("attention_mfma: `out` must be [n, nq, the values' width] in the dtype of q")
    if splits is None:
        # (keys of 128 with values of 32 to 128 in steps of 32 have the kernel of blocks that share a stage, and its rule
        # for splitting the keys; other pairs of widths stay on the kernel of single waves)
        tiles = d == 128 and dv % 32 == 0 and dv <= 128
        splits, chunk = attention_split(n_seqs, nkv, nq // nkv, max_q_len, max_kv_len, d if tiles or dv == d else 0)
    else:
        chunk = -(-(-(-max_kv_len // splits)) // 64) * 64
    target = _build.attn_target(d, dv)
    lib = library(target)
    ws_floats = lib.ia_attention_mfma_workspace(n, nq, splits)
    ws = torch.empty((ws_floats,), dtype=torch.float32, device=q.device) if ws_floats else None
    _check(lib.ia_attention_mfma(
        _p(out), _p(ws), _p(q), _p(k_cache), _p(v_cache), _p(block_table), _p(cu_tokens), _p(positions),
        n, seq_begin, n_seqs, token_begin, n_tokens, max_q_len, max_kv_len, block_table.shape[1], nq, nkv, d,
        page_size, int(window or 0), ctypes.c_float(scale), splits, chunk, int(bool(sink)), int(mask_chunk or 0), _p(sinks),
        int(keep_first), ctypes.c_float(softcap or 0.0), _stream()), target)
    return out


class DecodeCounters(dict):
    """The decode kernel's counters, an array a device: zero between calls (the kernel puts them back).  Calls that share them must follow
    each other (one stream, or a graph replayed on it), as an engine's steps do; every engine holds its own, so that two engines can
    run on two streams of a device."""

    dtype, what = torch.int32, "attention_decode_fused: the counters of the decode kernel"

    def __init__(self):
        super().__init__()
        self._outgrown: list = []                   # captured graphs may still hold their addresses: kept as long as this is

    def take(self, device: torch.device, needed: int) -> Optional[torch.Tensor]:
        """At least `needed` of them on `device` (None for none)."""
        if needed <= 0:
            return None
        key = device.index if device.index is not None else torch.cuda.current_device()
        have = self.get(key)
        if have is None or have.numel() < needed:
            if torch.cuda.is_current_stream_capturing():
                raise KernelError(f"{self.what} cannot be allocated under graph capture; run a step of this size once before capturing it")
            if have is not None:
                self._outgrown.append(have)
            have = torch.zeros((max(DECODE_COUNTERS_MIN, 2 * needed),), dtype=self.dtype, device=device)
            self[key] = have
        return have


_DECODE_COUNTERS = DecodeCounters()                 # of calls that bring none
DECODE_COUNTERS_MIN = 1 << 16


@functools.lru_cache(maxsize=4096)
def _decode_sizes(target: str, n: int, nq: int, nkv: int, splits: int) -> Tuple[int, int]:
    """(floats of workspace, counters) of a decode step."""
    lib = _raw_library(target)
    return lib.ia_attention_decode_workspace(n, nq, nkv, splits), lib.ia_attention_decode_counters(n, nq, nkv, splits)


def attention_decode_fused_fits(dtype: torch.dtype, d: int, page_size: int, rot: int, interleaved: bool,
                                has_rotation: bool, dv: Optional[int] = None) -> bool:
    """Whether decode steps can take `attention_decode_fused`: what the matrix-core kernel takes, keys' widths
    in steps of 64, and a rotation (if any) of the first features of a head in steps of 8, halves paired."""
    return (attention_mfma_fits(dtype, d, page_size, dv) and d % 64 == 0
            and (not has_rotation or (rot % 8 == 0 and 0 < rot <= d and not interleaved)))


def attention_decode_fused(qkv: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, positions: torch.Tensor,
                           cu_tokens: torch.Tensor, block_table: torch.Tensor, *, nq: int, nkv: int, d: int,
                           slots: Optional[torch.Tensor], q_norm_w: Optional[torch.Tensor],
                           k_norm_w: Optional[torch.Tensor], eps: float, add_one: bool,
                           cos: Optional[torch.Tensor], sin: Optional[torch.Tensor], max_kv_len: int,
                           window: Optional[int], scale: float, splits: Optional[int] = None,
                           seqs: Optional[Tuple[int, int]] = None, out: Optional[torch.Tensor] = None,
                           sink: bool = False, mask_chunk: Optional[int] = None, dv: Optional[int] = None,
                           offsets: Optional[Tuple[int, Optional[int], Optional[int]]] = None, rot: Optional[int] = None,
                           gate_off: Optional[int] = None, gate_per_head: bool = False,
                           counters: Optional[DecodeCounters] = None) -> torch.Tensor:
    """Decode steps (one token a request) in one kernel: per-head norm of q and k, rotation, the write
    of the new key and value at `slots` (None: the cache is only read) and the attention over the pages.
    `qkv` [n, (nq + 2 nkv) * d] is the projections' output; request s owns token s.  Returns [n, nq, d].
    Rows of other layouts: values of width `dv`, `offsets` = where the query, key and value heads begin in a row (the last two
    are None where nothing is written), `rot` = the first features of a head that rotate, and `gate_off` = where a row's gate values
    begin (one a feature of the joined heads, or `gate_per_head`): the output is times their sigmoid.  `counters`: those of the caller's
    stream (None: one set a device, for callers that use one stream)."""
    _dev(qkv, k_cache, v_cache, positions, cu_tokens, block_table, slots, q_norm_w, k_norm_w, cos, sin, out)
    _i32(positions, "positions"); _i32(cu_tokens, "cu_tokens"); _i32(block_table, "block_table")
    _f32(q_norm_w, "q_norm weight"); _f32(k_norm_w, "k_norm weight"); _f32(cos, "cos"); _f32(sin, "sin")
    n = qkv.shape[0]
    page_size = k_cache.shape[2]
    dv, rot = d if dv is None else dv, d if rot is None else rot
    _check_cache(k_cache, v_cache, nkv, page_size, d, qkv.dtype, "attention_decode_fused", dv)
    if not attention_decode_fused_fits(qkv.dtype, d, page_size, rot, False, cos is not None, dv):
        raise KernelError(f"attention_decode_fused: takes bfloat16, head sizes in steps of 64 and page sizes in "
                          f"steps of 16; got {qkv.dtype}, head size {d}, page size {page_size}")
    if offsets is None:
        offsets = (0, nq * d, (nq + nkv) * d)
        if qkv.dim() != 2 or qkv.shape[1] != (nq + nkv) * d + nkv * dv or nq % nkv:
            raise KernelError(f"attention_decode_fused: qkv has shape {tuple(qkv.shape)}, expected [n, {(nq + nkv) * d + nkv * dv}]")
    ld_ = qkv.shape[-1]
    q_off, k_off, v_off = offsets
    if (qkv.dim() != 2 or nq % nkv or ld_ % 4 or q_off % 4 or q_off < 0 or q_off + nq * d > ld_
            or (slots is not None and (k_off is None or v_off is None or k_off % 4 or k_off < 0 or k_off + nkv * d > ld_
                                       or v_off < 0 or v_off + nkv * dv > ld_))):
        raise KernelError(f"attention_decode_fused: heads at {offsets} of rows {tuple(qkv.shape)}")
    if gate_off is not None and (gate_off < 0 or gate_off + nq * (1 if gate_per_head else dv) > ld_ or (not gate_per_head and gate_off % 4)):
        raise KernelError(f"attention_decode_fused: gate values at {gate_off} of rows {tuple(qkv.shape)}")
    all_seqs = cu_tokens.numel() - 1
    seq_begin, n_seqs = seqs if seqs is not None else (0, all_seqs)
    if (positions.numel() != n or block_table.dim() != 2 or block_table.shape[0] < all_seqs or seq_begin < 0
            or seq_begin + n_seqs > all_seqs or seq_begin + n_seqs > n):
        raise KernelError("attention_decode_fused: positions, cu_tokens, block_table and the range do not fit the batch")
    if max_kv_len > block_table.shape[1] * page_size:
        raise KernelError(f"attention_decode_fused: max_kv_len {max_kv_len} does not fit {block_table.shape[1]} pages")
    for w, name in ((q_norm_w, "q_norm"), (k_norm_w, "k_norm")):
        if w is not None and w.numel() != d:
            raise KernelError(f"attention_decode_fused: {name} weight has {w.numel()} entries, head_dim is {d}")
    if (slots is not None and (q_norm_w is None) != (k_norm_w is None)) or (cos is None) != (sin is None):
        raise KernelError("attention_decode_fused: norm weights and angle tables come in pairs")
    if cos is not None and (cos.shape != (n, rot // 2) or sin.shape != cos.shape):
        raise KernelError(f"attention_decode_fused: rotary tables must be [{n}, {rot // 2}]")
    if slots is not None:
        _i32(slots, "slots")
        if slots.numel() != n:
            raise KernelError(f"attention_decode_fused: {slots.numel()} slots for {n} tokens")
    if out is None:
        out = torch.empty((n, nq, dv), dtype=qkv.dtype, device=qkv.device)
    elif tuple(out.shape) != (n, nq, dv) or out.dtype != qkv.dtype:
        raise KernelError("attention_decode_fused: `out` must be [n, nq, the values' width] in the dtype of qkv")
    if splits is None:
        splits, chunk = decode_shares(n_seqs, nkv, nq // nkv, max_kv_len, d, dv)
    else:
        chunk = -(-(-(-max_kv_len // splits)) // 32) * 32
    target = _build.attn_target(d, dv)
    lib = library(target)
    ws_floats, n_counters = _decode_sizes(target, n, nq, nkv, splits)
    ws = torch.empty((ws_floats,), dtype=torch.float32, device=qkv.device) if ws_floats else None
    taken = (_DECODE_COUNTERS if counters is None else counters).take(qkv.device, n_counters)
    _check(lib.ia_attention_mfma_decode_fused(
        _p(out), _p(ws), _p(qkv), _p(k_cache), _p(v_cache), _p(block_table), _p(cu_tokens), _p(positions), _p(slots),
        _p(q_norm_w), _p(k_norm_w), _p(cos), _p(sin), eps, int(add_one), ld_, q_off, k_off or 0, v_off or 0,
        rot if cos is not None else 0, _p(qkv) + 2 * gate_off if gate_off is not None else None, ld_, int(gate_per_head), n, seq_begin,
        n_seqs, seq_begin, n_seqs, max_kv_len, block_table.shape[1], nq, nkv, d, page_size, int(window or 0),
        scale, splits, chunk, int(bool(sink)), int(mask_chunk or 0), _p(taken),
        taken.numel() if taken is not None else 0, _stream()), target)
    return out


# ---- whole layers of decode steps of few rows ----------------------------------------------------

class RunWords(DecodeCounters):
    """The words through which the blocks of `layer_run` hand rows on, with its counter; as the decode kernel's counters, an engine's own.
    A block that waits for another's words gives up after `polls` reads, so that no launch hangs; the launch's rows, and the keys and values that it
    caches, are then no numbers.  No wait of a sound launch comes near the limit: `check`, which an engine calls wherever it has waited for the
    device, makes an error of one that did."""
    dtype, what = torch.int64, "layer_run: the words of runs of layers"
    POLLS = 1 << 20                                 # (seconds)

    def __init__(self):
        super().__init__()
        self.polls = self.POLLS
        self.given_up = torch.zeros((1,), dtype=torch.int32, pin_memory=torch.cuda.is_available())      # (the kernel writes it from the device)

    def check(self) -> None:
        """Raises where a launch that has ended gave a wait up, once for all launches since the last check."""
        if self.given_up.item():
            self.given_up.zero_()
            raise KernelError("layer_run: a decode step's blocks waited in vain for each other's rows; the logits of the steps since the last "
                              "check, and the keys and values that these cached, are void")


RUN_MAX_ROWS = 8
RUN_SHARED_BYTES = 160 * 1024 - 64


def run_shares(max_kv_len: int) -> Tuple[int, int]:
    """(shares, keys of a share) of a row's keys in `layer_run`."""
    chunk = 512 * max(1, -(-max_kv_len // (512 * 32)))
    return -(-max_kv_len // chunk), chunk


def layer_run_fits(rows: int, width: int, ff: int, nq: int, nkv: int, page_size: int) -> bool:
    """Whether `layer_run` takes steps of these sizes: what a wave loads at once divides the inner widths, and a step's widest rows
    fit a compute unit's shared memory."""
    return (1 <= rows <= RUN_MAX_ROWS and page_size == 16 and width % 512 == 0 and width <= 6144 and ff % 512 == 0 and nq % nkv == 0
            and nq // nkv <= 8 and nq % 4 == 0 and rows * (max(width, ff, nq * 128) * 2 + 384) <= RUN_SHARED_BYTES)


def layer_run_aligned(layers: Sequence[Sequence[torch.Tensor]]) -> bool:
    """Whether `layer_run` can read these layers' arrays: weights and caches 16 bytes at a time, the norms' weights 8."""
    wide = pairs = 0
    for qkv, o, gate_up, down, norm1, norm2, q_norm, k_norm, k, v in layers:
        wide |= qkv.data_ptr() | o.data_ptr() | gate_up.data_ptr() | down.data_ptr() | k.data_ptr() | v.data_ptr()
        pairs |= norm1.data_ptr() | norm2.data_ptr() | q_norm.data_ptr() | k_norm.data_ptr()
    return wide % 16 == 0 and pairs % 8 == 0


def layer_run_pays(rows: int, width: int, ff: int, nq: int, nkv: int, max_kv_len: int, layers: int = 6) -> bool:
    """Whether a step of these sizes is faster by `layer_run` over a run of `layers` than by five kernels a layer.  What it gains is a layer's launches,
    first bytes and last sums.  They weigh less the larger the weights are, the more rows every block fetches for itself, and the more bytes of
    keys and values there are, which the decode attention walks with twice the waves a compute unit.  Of 1,150 sizes of 29 shapes it takes 900,
    1.3 times as fast in the mean, the worst 0.98 (both ways replayed from graphs in turn; us a layer, five kernels / a run).
    Rows.  Weights up to 128 MiB: 0.6B shape, 700 keys, 1 row 31 / 15, 8 rows 36 / 23; 1.7B shape, 8 rows 51 / 39.  Up to 256 MiB: 4B shape, 4 rows
    68 / 57, 6 rows 70 / 64 (one layer 0.87 to 1.03), 8 rows 72 / 69 (1.00 to 1.08 from six layers on, of one to four layers 0.84 to 0.99: a run's
    first layers gain less than those behind them); with more than 8 key heads attention alone is more blocks than units from 6 rows on (width 2,048, 32 key heads, 5 rows 66 / 62,
    6 rows 68 / 68, 8 rows 74 / 76); widths of 3,072 and 3,584, of which a wave takes six or seven loads and only four ahead of its wait: 3 rows 60 /
    58, 4 rows 61 / 67.  Up to 512 MiB: 8B shape 3 rows 91 / 78, 4 rows 92 / 94, 6 rows 95 / 105.  Beyond: 14B shape 2 rows 142 / 126, 32B shape 199 / 184.
    Keys.  One row: 0.6B shape at 45,000 keys 59 / 50; 32 key heads of width 2,048 at 16,384 0.995 of the speed, at 33,000 1.065, at 45,000 1.05; 40 of
    width 5,120 at 24,000 1.08.  More: 16 key heads, 4 rows at 8,192 1.08 to 1.11, 5 rows 0.99 to 1.00, 2 rows at 16,384 0.96 to 1.00; 32 key heads,
    2 rows at 8,192 1.03 to 1.07, 3 rows at 11,000 0.92; 40 of width 5,120, 2 rows at 8,192 1.02, at 12,000 0.97."""
    weights = 2 * (2 * (nq + nkv) * 128 * width + 3 * width * ff)
    bytes_of_keys = 512 << 10                       # (rows x keys x key heads)
    if weights <= 128 << 20:
        most, keys = 8, 44 << 10
    elif weights <= 256 << 20:
        most, keys = (3 if 6 <= width // 512 < 8 else 4 if layers < 2 else 5 if nkv > 8 else 6 if layers < 6 else 8), 44 << 10
    elif weights <= 512 << 20:
        most, keys = 3, 20 << 10
    else:
        most, keys, bytes_of_keys = 2, 24 << 10, 640 << 10
    return (rows <= most and rows * max_kv_len <= keys
            and (rows == 1 or (rows * max_kv_len * nkv <= bytes_of_keys and (nkv <= 8 or max_kv_len <= 12 << 10))))


def layer_run(x: torch.Tensor, layers: Sequence[Sequence[torch.Tensor]], words: RunWords, positions: torch.Tensor, slots: torch.Tensor,
              block_table: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, *, nq: int, nkv: int, ff: int, max_kv_len: int,
              eps: Tuple[float, float, float], add_one: Tuple[bool, bool, bool], scale: float) -> torch.Tensor:
    """A run of whole layers over the stream `x` [rows, width], in place: `layers` holds each layer's [q | k | v], o, [gate; up] and down
    weights, the norms' weights of the stream (two) and of the heads (q, k), and its arrays of keys and values; `eps` and `add_one` are
    those of the three kinds of norms.  Row i is the newest token of request i."""
    _dev(x, positions, slots, block_table, cos, sin)
    _i32(positions, "positions"); _i32(slots, "slots"); _i32(block_table, "block_table")
    _f32(cos, "cos"); _f32(sin, "sin")
    rows, width = x.shape
    if x.dtype != torch.bfloat16 or not layers:
        raise KernelError("layer_run: bfloat16 rows and one layer or more")
    page_size = layers[0][8].shape[2]
    if not layer_run_fits(rows, width, ff, nq, nkv, page_size):
        raise KernelError(f"layer_run: {rows} rows of {width}, feed-forward {ff}, {nq} and {nkv} heads, pages of {page_size}")
    shapes = ([((nq + 2 * nkv) * 128, width), (width, nq * 128), (2 * ff, width), (width, ff)], [width, width, 128, 128])
    for of in layers:
        _dev(*of)
        if any(t.dtype != torch.bfloat16 or tuple(t.shape) != want for t, want in zip(of[:4], shapes[0])):
            raise KernelError(f"layer_run: weights {[tuple(t.shape) for t in of[:4]]}, expected bfloat16 {shapes[0]}")
        for t, want in zip(of[4:8], shapes[1]):
            _f32(t, "norm weight")
            if t.numel() != want:
                raise KernelError(f"layer_run: a norm weight of {t.numel()} entries, expected {want}")
        _check_cache(of[8], of[9], nkv, page_size, 128, x.dtype, "layer_run", 128)
    if (positions.numel() != rows or slots.numel() != rows or block_table.dim() != 2 or block_table.shape[0] < rows
            or cos.shape != (rows, 64) or sin.shape != cos.shape or not 0 < max_kv_len <= block_table.shape[1] * page_size):
        raise KernelError("layer_run: positions, slots, block table and angles do not fit the rows")
    splits, chunk = run_shares(max_kv_len)
    lib = library()
    space = words.take(x.device, int(lib.ia_layer_run_words(rows, width, ff, nq, nkv, splits)))
    most = lib.ia_layer_run_layers()
    for lo in range(0, len(layers), most):
        of = layers[lo:lo + most]
        table = (ctypes.c_void_p * (10 * len(of)))(*[t.data_ptr() for layer in of for t in layer])
        _check(lib.ia_layer_run(
            _p(x), ctypes.addressof(table), len(of), _p(space), space.numel(), _p(words.given_up), words.polls, _p(positions), _p(slots),
            _p(block_table), _p(cos), _p(sin), rows, width, ff, nq, nkv, page_size, block_table.shape[1], max_kv_len, splits, chunk, *eps, *(int(o) for o in add_one), scale, _stream()))
    return x


# ---- matrix products --------------------------------------------------------------------------

# Beyond this many rows (one tile of MFMA columns) other kernels read the weights faster.  Up to 16 rows the
# skinny products also take over the sums and norms of the residual stream; a decode step at a context of 2,048
# and the sizes of an 8 B model takes 5.02 ms with 12 requests, 5.20 with 13 and 5.22 with 16 (5.54 and 5.44 with
# the vendor's GEMM and norm kernels of their own from 13 rows on; at the 14B shape 9.7 against 10.9 ms at 14 rows).
SKINNY_MAX_ROWS = 16


# Who multiplies more bfloat16 rows than the skinny kernel takes: "library" (the vendor's GEMM, as the reference's
# products go to cuBLAS) or "own" (the tiled matrix-core kernel of this package, where the width is a multiple of
# 64).  The library is faster at the sizes of an 8 B model (2,048 rows: 84, 60, 335 with SiLU and 168 us for qkv, o,
# gate|up and down against 125, 119, 435 and 323 us), so it is the default; INFERRS_AMD_LARGE_PRODUCTS=own
# runs the model without it.
LARGE_PRODUCTS = os.environ.get("INFERRS_AMD_LARGE_PRODUCTS", "library")


# How the vendor's GEMM is called: "direct" (hipBLASLt through this package's own entry point, which keeps descriptors,
# layouts and the library's choice of kernel for every shape: 7 us of host time a product) or "torch" (`F.linear`:
# 18 us a product whatever its size, more than the GPU needs for the products of a small model).  "direct" falls back
# to "torch", with a warning, where the library cannot be opened.
VENDOR_GEMM = os.environ.get("INFERRS_AMD_VENDOR_GEMM", "direct")
VENDOR_WORKSPACE_BYTES = 128 << 20
_VENDOR_STATE: Dict[str, object] = {}


def _vendor_library_path() -> Optional[str]:
    """The hipBLASLt that this process has loaded (torch brings its own copy), else torch's, else the system's."""
    try:
        with open("/proc/self/maps") as f:
            for line in f:
                if "libhipblaslt.so" in line:
                    return line.split(None, 5)[-1].strip()
    except OSError:
        pass
    for path in (os.path.join(os.path.dirname(torch.__file__), "lib", "libhipblaslt.so"), "/opt/rocm/lib/libhipblaslt.so"):
        if os.path.exists(path):
            return path
    return None


def _vendor_direct() -> bool:
    if VENDOR_GEMM not in ("direct", "torch"):
        raise KernelError(f"INFERRS_AMD_VENDOR_GEMM / ops.VENDOR_GEMM: 'direct' or 'torch', not {VENDOR_GEMM!r}")
    if VENDOR_GEMM == "torch":
        return False
    if "ready" not in _VENDOR_STATE:
        path = _vendor_library_path()
        lib = _raw_library()
        ok = path is not None and lib.ia_vendor_gemm_init(path.encode()) == 0
        if not ok:
            import logging
            logging.getLogger("inferrs_amd").warning(
                "the vendor's GEMM library could not be opened directly (%s): its products go through torch",
                lib.ia_last_error().decode() if path is not None else "libhipblaslt.so not found")
        _VENDOR_STATE["ready"] = ok
    return bool(_VENDOR_STATE["ready"])


def vendor_gemm_bf16(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x [m, k] . w[n, k]^T in bfloat16 through the vendor's GEMM library."""
    if not _vendor_direct() or x.shape[0] == 0:
        return torch.nn.functional.linear(x, w)
    _dev(x, w)
    m, k = x.shape
    n = w.shape[0]
    if w.shape[1] != k or x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16:
        raise KernelError(f"vendor_gemm: x {tuple(x.shape)} {x.dtype} does not fit w {tuple(w.shape)} {w.dtype}")
    if not (x.is_contiguous() and w.is_contiguous()):
        raise KernelError("vendor_gemm: operands must be contiguous")
    key = ("workspace", x.device.index)
    ws = _VENDOR_STATE.get(key)
    if ws is None:
        if torch.cuda.is_current_stream_capturing():
            # (the library's handle and the workspace are made outside a capture: a product that is the first of its
            # process and is being captured goes through torch)
            return torch.nn.functional.linear(x, w)
        ws = _VENDOR_STATE[key] = torch.empty((VENDOR_WORKSPACE_BYTES,), dtype=torch.uint8, device=x.device)
        warm = torch.zeros((16, 64), dtype=torch.bfloat16, device=x.device)
        if _raw_library().ia_vendor_gemm_bf16(_p(torch.empty((16, 16), dtype=torch.bfloat16, device=x.device)), _p(warm),
                                              _p(warm), 16, 16, 64, _p(ws), ws.numel(), _stream()) == 1:
            _check(1)
    refused = _VENDOR_STATE.setdefault("refused", set())
    if (m, n, k) in refused:
        return torch.nn.functional.linear(x, w)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
    code = _raw_library().ia_vendor_gemm_bf16(_p(out), _p(x), _p(w), m, n, k, _p(ws), ws.numel(), _stream())
    if code == 2:                                    # the library's search names no kernel for this shape (an odd k)
        refused.add((m, n, k))
        return torch.nn.functional.linear(x, w)
    _check(code)
    return out


def _own_large(x: torch.Tensor, w: torch.Tensor) -> bool:
    if LARGE_PRODUCTS not in ("library", "own"):
        raise KernelError(f"INFERRS_AMD_LARGE_PRODUCTS / ops.LARGE_PRODUCTS: 'library' or 'own', not {LARGE_PRODUCTS!r}")
    return (LARGE_PRODUCTS == "own" and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.shape[1] % 64 == 0
            and x.is_contiguous() and w.is_contiguous())


def gemm_mfma_bf16(x: torch.Tensor, w: torch.Tensor, dual: bool = False, activation: str = "silu") -> torch.Tensor:
    """x [m, k] . w[n, k]^T in bfloat16 by the tiled matrix-core kernel (k a multiple of 64); with `dual`
    w is [gate; up] and the result act(x . gate^T) * (x . up^T)."""
    _dev(x, w)
    m, k = x.shape
    rows, k2 = w.shape
    if k2 != k or x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or k % 64 or (dual and rows % 2):
        raise KernelError(f"gemm_mfma: x {tuple(x.shape)} {x.dtype} does not fit w {tuple(w.shape)} {w.dtype}")
    if not (x.is_contiguous() and w.is_contiguous()):
        raise KernelError("gemm_mfma: operands must be contiguous")
    n = rows // 2 if dual else rows
    out = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
    if m:
        _check(library().ia_gemm_mfma_bf16(_p(out), _p(x), _p(w), m, n, k, activation_code(activation) if dual else 0,
                                           _stream()))
    return out


def gemm_tiled(x: torch.Tensor, w: torch.Tensor, out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    _dev(x, w)
    m, k = x.shape
    n, k2 = w.shape
    if k != k2 or x.dtype != w.dtype:
        raise KernelError(f"gemm: x {tuple(x.shape)} {x.dtype} does not fit w {tuple(w.shape)} {w.dtype}")
    out_dtype = out_dtype or x.dtype
    out = torch.empty((m, n), dtype=out_dtype, device=x.device)
    _check(library().ia_gemm_tiled(_p(out), _p(x), _p(w), m, n, k, _dt(x), _DT[out_dtype], _stream()))
    return out


def _skinny_bias(bias: Optional[torch.Tensor], rows: int) -> None:
    if bias is not None and (bias.dtype != torch.bfloat16 or bias.numel() != rows or not bias.is_cuda
                             or not bias.is_contiguous()):
        raise KernelError(f"gemm_skinny: the bias must be a contiguous bfloat16 vector of {rows} entries on the GPU")


def gemm_skinny_bf16(x: torch.Tensor, w: torch.Tensor, out_dtype: torch.dtype = torch.bfloat16,
                     dual: bool = False, activation: str = "silu", bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x [m, k] . w[n, k]^T (+ bias) on the matrix cores, made for few rows.  `dual`: w is [gate; up]
    stacked along its rows and the result is act(x . gate^T + bias[:n]) * (x . up^T + bias[n:])."""
    _dev(x, w)
    _skinny_bias(bias, w.shape[0])
    m, k = x.shape
    n, k2 = w.shape
    if k != k2 or x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16:
        raise KernelError(f"gemm_skinny: x {tuple(x.shape)} {x.dtype} does not fit w {tuple(w.shape)} {w.dtype}")
    if dual:
        if n % 2:
            raise KernelError(f"gemm_skinny: a stacked [gate; up] weight needs an even row count, got {n}")
        n //= 2
    out = torch.empty((m, n), dtype=out_dtype, device=x.device)
    _check(library().ia_gemm_skinny_bf16(_p(out), _p(x), _p(w), _p(bias), m, n, k, _DT[out_dtype],
                                         activation_code(activation) if dual else 0, _stream()))
    return out


def skinny_fits(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (x.dtype == torch.bfloat16 and x.shape[1] % 8 == 0 and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def fill_normal(shape, seed: int, mean: float, std: float, dtype: torch.dtype, device) -> torch.Tensor:
    """A tensor of mean + std * N(0, 1), element i a function of (seed, i) alone; the same values
    as the host fill of `inferrs_amd.weights.random_init`."""
    require_gpu()
    out = torch.empty(tuple(shape), dtype=dtype, device=device)
    _check(library().ia_fill_normal(_p(out), ctypes.c_longlong(out.numel()), ctypes.c_ulonglong(seed & (2**64 - 1)),
                                    ctypes.c_double(mean), ctypes.c_double(std), _dt(out), _stream()))
    return out


def stream_read(x: torch.Tensor, blocks: int = 4096) -> torch.Tensor:
    """Reads all of `x` once (a multiple of 16 bytes), a contiguous range a block: the measurement script times it for
    the memory's practical read rate.  (The returned words are scratch.)"""
    _dev(x)
    nbytes = x.numel() * x.element_size()
    out = torch.zeros((blocks,), dtype=torch.int32, device=x.device)
    _check(library().ia_stream_read(_p(out), _p(x), ctypes.c_longlong(nbytes), blocks, _stream()))
    return out


def widen(x: torch.Tensor) -> torch.Tensor:
    """bfloat16 -> float32, exactly."""
    _dev(x)
    if x.dtype != torch.bfloat16:
        raise KernelError(f"widen: takes bfloat16, got {x.dtype}")
    out = torch.empty(x.shape, dtype=torch.float32, device=x.device)
    _check(library().ia_widen_bf16(_p(out), _p(x), ctypes.c_longlong(x.numel()), _stream()))
    return out


# ---- a residual stream around the skinny product ---------------------------------------------
# Decode steps have a few rows, and a kernel of its own that adds a product to the stream and norms the
# sum is all launch and latency.  The product before such a norm can add itself to the stream
# (`linear_add`): it leaves every row's sum of squares, block by block, and the new rows times the
# norm's weight; the product after the norm (`linear` / `gated_silu_linear` given `NormedRows`) takes
# those rows and multiplies its sums by the row's scale, rsqrt(mean of squares + eps).

STREAM_MAX_ROWS = 16          # rows up to which the products take over the sums and norms of a step


class Added:
    """What a part returns instead of its output when it has added it to the step's stream itself:
    `sums` [rows, blocks] are the partial sums of squares of the stream's new rows and `scaled` the
    new rows times the weight of `norm` (the norm part that comes next), or None."""
    __slots__ = ("sums", "scaled", "norm")

    def __init__(self, sums: torch.Tensor, scaled: Optional[torch.Tensor] = None, norm=None):
        self.sums, self.scaled, self.norm = sums, scaled, norm


class NormedRows:
    """Rows of a stream `x` whose norm, rmsnorm(x; weight, eps), is left to the product that reads them:
    `scaled` = x * weight (rounded once) and `sums` [rows, blocks] the rows' sums of squares."""
    __slots__ = ("x", "scaled", "sums", "weight", "eps", "add_one")

    def __init__(self, x: torch.Tensor, scaled: torch.Tensor, sums: torch.Tensor, weight: torch.Tensor, eps: float,
                 add_one: bool):
        self.x, self.scaled, self.sums, self.weight = x, scaled, sums, weight
        self.eps, self.add_one = float(eps), bool(add_one)

    @property
    def shape(self):
        return self.x.shape

    @property
    def dtype(self):
        return self.x.dtype

    def materialize(self) -> torch.Tensor:
        return rmsnorm(self.x, self.weight, self.eps, self.add_one)


def _stream_product(x: torch.Tensor, w: torch.Tensor, n: int, out_dtype, dual: bool, resid=None, sums_out=None,
                    scaled_out=None, next_w=None, add_one: bool = False, sums_in=None, eps: float = 0.0,
                    activation: str = "silu", bias: Optional[torch.Tensor] = None):
    m, k = x.shape
    _skinny_bias(bias, w.shape[0])
    out = None if resid is not None else torch.empty((m, n), dtype=out_dtype, device=x.device)
    _check(library().ia_gemm_skinny_stream(
        _p(out), _p(x), _p(w), _p(bias), m, n, k, _DT[out_dtype], activation_code(activation) if dual else 0, _p(resid),
        _p(sums_out), _p(scaled_out), _p(next_w),
        int(add_one), _p(sums_in), sums_in.shape[1] if sums_in is not None else 0, ctypes.c_float(eps), _stream()))
    return out


def _takes_normed_rows(x: NormedRows, w: torch.Tensor, n: int) -> bool:
    m, k = x.scaled.shape
    return (m <= SKINNY_MAX_ROWS and x.scaled.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and w.shape[1] == k
            and skinny_fits(x.scaled, w) and n < 65536 and x.sums.dtype == torch.float32 and x.sums.shape[0] == m
            and x.sums.is_contiguous() and x.scaled.is_contiguous())


def linear_add(x: torch.Tensor, w: torch.Tensor, resid: torch.Tensor, next_norm=None,
               bias: Optional[torch.Tensor] = None):
    """resid += x . w^T (+ bias) in place, as `add_rmsnorm` would add the product (rounded, then summed in 32-bit
    and rounded), by the skinny kernel itself.  Returns (sums, scaled): the partial sums of squares of the
    new rows [rows, blocks], and the new rows times the weight of `next_norm` (a norm part with `weight`
    and `add_one`; None: no such rows); or None when this product cannot (the caller then forms it and
    lets the norm add it)."""
    m, k = x.shape
    n = w.shape[0]
    if (m > SKINNY_MAX_ROWS or m == 0 or x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or w.shape[1] != k
            or not skinny_fits(x, w) or n >= 65536 or resid.dtype != torch.bfloat16 or tuple(resid.shape) != (m, n)
            or not resid.is_contiguous() or (bias is not None and bias.dtype != torch.bfloat16)):
        return None
    next_w = getattr(next_norm, "weight", None)
    if next_w is not None and (next_w.dtype != torch.float32 or next_w.numel() != n):
        next_w = None
    _dev(x, w, resid, next_w)
    sums = torch.empty((m, library().ia_gemm_skinny_blocks(n)), dtype=torch.float32, device=x.device)
    scaled = torch.empty_like(resid) if next_w is not None else None
    _stream_product(x, w, n, torch.bfloat16, False, resid=resid, sums_out=sums, scaled_out=scaled, next_w=next_w,
                    add_one=bool(getattr(next_norm, "add_one", False)), bias=bias)
    return sums, scaled


# ---- products of 17 to 128 rows ------------------------------------------------------------------
# Decode steps of many requests and short prompt portions: still bound by reading the weights once, which the vendor's
# GEMM does at 2 to 3.4 TB/s and the kernel of gemm_mid.hip faster.  (Sizes of an 8B model, a prompt of 128 tokens, the four
# products of a layer inside the model: 129 us against 174 through the vendor's GEMM; of 65 tokens: 108 against 182.)  Weights with few rows (the output projection, the
# feed-forward's second product) are split along k between blocks, and the splits' sums are added up by the reader:
# `Partials` stands for a product in that state.

MID_MAX_ROWS = 128            # rows up to which the products of gemm_mid.hip take over from the vendor's GEMM
# Rows from which a layer's products go to gemm_mid.hip, with kernels of their own for the sums of the splits and the norms,
# instead of the skinny products that take over the stream's sums and norms: None = by the rule of `mid_from_rows`.
MID_FROM_ROWS: Optional[int] = None
MID_MIN_ROWS = 5              # fewest rows for which a split product is worth the kernel that adds it up


def mid_from_rows(width: int) -> int:
    """Rows of a step from which the products of a model of this width (the residual stream's) run on gemm_mid.hip.
    Measured, decode steps at a context of 700, the step's time on gemm_mid.hip over that with the skinny products: width 1,024
    (0.6B shape) 8 rows 1.18, 12 rows 1.15, 16 rows 1.11; 2,048 (1.7B) 8 rows 1.06, 12 rows 1.02, 16 rows 0.97; 4,096 (8B) 8 rows 1.04,
    10 rows 1.01, 12 rows 1.00, 16 rows 0.99.  A width that is no power of two leaves the skinny product's waves uneven shares of k and
    blocks that are no whole tiles: 2,560 (4B) 5 rows 1.00, 6 rows 0.98, 10 rows 0.93, 16 rows 0.89; 5,120 (14B) 5 rows 1.03, 6 rows 1.00,
    8 rows 0.99, 16 rows 0.89.  (Narrower powers of two were not measured and stay at 9.)"""
    if MID_FROM_ROWS is not None:
        return MID_FROM_ROWS
    if width & (width - 1) == 0:
        return 9 if width < 1024 else 17 if width < 2048 else 13
    return MID_MIN_ROWS if width < 4096 else 6
# [gate; up] weights beyond this many bytes go to the vendor's GEMM and the SiLU kernel also at 17 to 64 rows.  Measured at 32
# rows (kernel after kernel, launch gaps included): 2 x 12,288 x 4,096 (201 MB) 49 us here against 49 + 5 us there,
# 2 x 25,600 x 5,120 (524 MB) 125 us here against 96 + 5 us there; the plain products are faster here at every size
# (5,120 x 25,600: 57 us against 147).
MID_DUAL_MAX_BYTES = 256 << 20
MID_PRODUCTS = os.environ.get("INFERRS_AMD_MID_PRODUCTS", "own")      # "own" or "library"


class Partials:
    """A product [rows, features] as the 32-bit sums of each split of k, `parts` [splits, rows, features]; whoever
    needs it adds them up in the order of the splits (`materialize()`, or `add_rmsnorm_partials`)."""
    __slots__ = ("parts",)

    def __init__(self, parts: torch.Tensor):
        self.parts = parts

    @property
    def shape(self):
        return self.parts.shape[1:]

    def materialize(self) -> torch.Tensor:
        splits, m, n = self.parts.shape
        out = torch.empty((m, n), dtype=torch.bfloat16, device=self.parts.device)
        _check(library().ia_sum_partials(_p(out), _p(self.parts), splits, m, n, _stream()))
        return out


def mid_fits(x: torch.Tensor, w: torch.Tensor, few_rows: bool = False) -> bool:
    """Whether x . w^T goes to gemm_mid.hip: from `mid_from_rows(k)` to `MID_MAX_ROWS` rows (`few_rows`: from 1 row on)."""
    if MID_PRODUCTS not in ("own", "library"):
        raise KernelError(f"INFERRS_AMD_MID_PRODUCTS / ops.MID_PRODUCTS: 'own' or 'library', not {MID_PRODUCTS!r}")
    return (MID_PRODUCTS == "own" and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
            and (1 if few_rows else mid_from_rows(x.shape[1])) <= x.shape[0] <= MID_MAX_ROWS
            and x.shape[1] % 128 == 0 and w.shape[1] == x.shape[1]
            and x.is_contiguous() and w.is_contiguous() and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def gemm_mid_bf16(x: torch.Tensor, w: torch.Tensor, out_dtype: torch.dtype = torch.bfloat16, dual: bool = False,
                  partial: bool = False, sums_in: Optional[torch.Tensor] = None, eps: float = 0.0,
                  activation: str = "silu"):
    """x [m, k] . w[n, k]^T for 1 to 128 bfloat16 rows and k a multiple of 128 (gemm_mid.hip).  `dual`: w = [gate; up],
    the result act(x . gate^T) * (x . up^T).  `partial`: the result stays split along k, as `Partials` (a weight that
    needs no split gives a plain tensor).  `sums_in` [m, blocks] (up to 16 rows): the rows are a norm's input times its
    weight and these their sums of squares; every sum is multiplied by the row's rsqrt(mean of squares + eps)."""
    _dev(x, w)
    m, k = x.shape
    rows, k2 = w.shape
    if (k2 != k or x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or k % 128 or not (1 <= m <= MID_MAX_ROWS)
            or (dual and (rows % 2 or partial or out_dtype != torch.bfloat16))):
        raise KernelError(f"gemm_mid: x {tuple(x.shape)} {x.dtype} does not fit w {tuple(w.shape)} {w.dtype} "
                          f"(1 to {MID_MAX_ROWS} rows, k a multiple of 128)")
    n = rows // 2 if dual else rows
    lib = library()
    act = activation_code(activation) if dual else 0
    if partial:
        splits = lib.ia_gemm_mid_splits(n, k)
        if splits > 1 and (m * n) % 4 == 0:
            parts = torch.empty((splits, m, n), dtype=torch.float32, device=x.device)
            _check(lib.ia_gemm_mid_bf16(_p(parts), _p(x), _p(w), m, n, k, 2, 0, _stream()))
            return Partials(parts)
    out = torch.empty((m, n), dtype=out_dtype, device=x.device)
    if sums_in is not None:
        _dev(sums_in); _f32(sums_in, "sums of squares")
        if partial or m > 16 or sums_in.dim() != 2 or sums_in.shape[0] != m or not sums_in.is_contiguous():
            raise KernelError(f"gemm_mid: sums of squares {tuple(sums_in.shape)} for {m} rows (up to 16, whole sums)")
        _check(lib.ia_gemm_mid_bf16_scaled(_p(out), _p(x), _p(w), m, n, k, 0 if out_dtype == torch.bfloat16 else 1,
                                           act, _p(sums_in), sums_in.shape[1], ctypes.c_float(eps), _stream()))
        return out
    _check(lib.ia_gemm_mid_bf16(_p(out), _p(x), _p(w), m, n, k, 0 if out_dtype == torch.bfloat16 else 1,
                                act, _stream()))
    return out


# ---- products of 129 to 2,048 rows ---------------------------------------------------------------
# Steps with prompt portions: gemm_wide.hip splits k between blocks where the vendor's GEMM leaves the chip half empty (its
# header has the figures; which product goes there is asked of ia_gemm_wide_norm_fits, _rope_fits and _dual_fits).
WIDE_MAX_ROWS = 2048


def wide_fits(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether gemm_wide.hip takes x . w^T (beyond the rows of gemm_mid.hip, up to `WIDE_MAX_ROWS`); not where the switches ask
    for the vendor's GEMM or for the tiled kernel of gemm_mfma.hip throughout."""
    return (MID_PRODUCTS == "own" and LARGE_PRODUCTS == "library" and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
            and MID_MAX_ROWS < x.shape[0] <= WIDE_MAX_ROWS and x.shape[1] % 64 == 0 and w.shape[1] == x.shape[1]
            and w.shape[0] % 4 == 0 and x.is_contiguous() and w.is_contiguous() and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def gemm_wide_bf16(x: torch.Tensor, w: torch.Tensor, dual: bool = False, partial: bool = False, activation: str = "silu"):
    """x [m, k] . w[n, k]^T in bfloat16 (k a multiple of 64, n of 4); `dual` and `partial` as `gemm_mid_bf16` has them."""
    _dev(x, w)
    m, k = x.shape
    rows, k2 = w.shape
    if (k2 != k or x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or m < 1 or k % 64 or rows % (8 if dual else 4)
            or (dual and partial) or not (x.is_contiguous() and w.is_contiguous())):
        raise KernelError(f"gemm_wide: x {tuple(x.shape)} {x.dtype} does not fit w {tuple(w.shape)} {w.dtype}")
    n = rows // 2 if dual else rows
    lib = library()
    if partial:
        splits = lib.ia_gemm_wide_splits(m, n, k)
        if splits > 1:
            parts = torch.empty((splits, m, n), dtype=torch.float32, device=x.device)
            _check(lib.ia_gemm_wide_bf16(_p(parts), _p(x), _p(w), m, n, k, 2, 0, _stream()))
            return Partials(parts)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
    _check(lib.ia_gemm_wide_bf16(_p(out), _p(x), _p(w), m, n, k, 0, activation_code(activation) if dual else 0, _stream()))
    return out


def gemm_wide_rows(x: torch.Tensor, w: torch.Tensor, act: int = 0) -> torch.Tensor:
    """x [m, k] . w[n, k]^T in bfloat16 with an activation of `state.activation` (0: none) over the rounded result (k a multiple of 64, n of 4)."""
    _dev(x, w)
    m, k = x.shape
    n, k2 = w.shape
    if (k2 != k or x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or m < 1 or k % 64 or n % 4
            or not (x.is_contiguous() and w.is_contiguous())):
        raise KernelError(f"gemm_wide_rows: x {tuple(x.shape)} {x.dtype} does not fit w {tuple(w.shape)} {w.dtype}")
    out = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
    _check(library().ia_gemm_wide_rows_bf16(_p(out), _p(x), _p(w), m, n, k, act, _stream()))
    return out


def activated_linear(x, w: torch.Tensor, act: int) -> torch.Tensor:
    """An activation of `state.activation` over x . w^T: inside the product where that is faster."""
    if isinstance(x, torch.Tensor) and _wide_takes("act", x, w):
        return gemm_wide_rows(x, w, act)
    return activation(linear(x, w), act)


def _wide_takes(rule: str, x: torch.Tensor, w: torch.Tensor) -> bool:
    return (x.shape[0] > MID_MAX_ROWS and x.dim() == 2 and w.shape[0] % 4 == 0 and _wide_pays(rule, x.shape[0], w.shape[0], x.shape[1])
            and wide_fits(x, w))


@functools.lru_cache(maxsize=4096)
def _wide_pays(reader: str, m: int, n: int, k: int) -> bool:
    """gemm_wide.hip's rule for `m` rows, `n` features and k ahead of a reader ("norm", "rope", or "dual": [gate; up] of n features
    each).  A rule follows from these sizes alone and is asked three times a layer, so its answers are kept: a step that the host
    bounds waits for each (0.7 to 0.9 us through ctypes; a product that stays with the vendor's GEMM 4.6 us of asking -> 0.6)."""
    return m <= WIDE_MAX_ROWS and bool(getattr(library(), f"ia_gemm_wide_{reader}_fits")(m, n, k))


def linear_partials(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None, own_rows: bool = False):
    """x . w^T for a reader that takes `Partials`, split along k where the weight has few rows: the norm that adds the product to
    the stream, or (`own_rows`) the kernel that norms and turns queries and keys.  None where `linear` is faster, or where
    neither gemm_mid.hip (up to `MID_MAX_ROWS` rows) nor gemm_wide.hip (up to `WIDE_MAX_ROWS`) takes these operands, a bias among
    them: the caller then forms the whole product, and `linear` adds the bias."""
    # (up to MID_MAX_ROWS rows: who asks ahead of the norm is in a step whose products go to gemm_mid.hip, the rule has been asked with
    # the stream's width, and a product of another width follows it; with `own_rows` the width of the rows themselves decides)
    if bias is not None or not isinstance(x, torch.Tensor):
        return None
    m, k = x.shape
    if m <= MID_MAX_ROWS:
        if m >= MID_MIN_ROWS and mid_fits(x, w, few_rows=not own_rows):
            return gemm_mid_bf16(x, w, partial=True)
    elif _wide_pays("rope" if own_rows else "norm", m, w.shape[0], k) and wide_fits(x, w):
        return gemm_wide_bf16(x, w, partial=True)
    return None


def add_rmsnorm_partials(x: torch.Tensor, delta: Partials, w: torch.Tensor, eps: float, add_one: bool = False) -> torch.Tensor:
    """x += delta in place, delta's splits added up and rounded to bfloat16 first (as a stored product would be);
    returns rmsnorm(x)."""
    parts = delta.parts
    _dev(x, parts, w); _f32(w, "norm weight")
    splits, rows, cols = parts.shape
    if x.dtype != torch.bfloat16 or tuple(x.shape) != (rows, cols) or w.numel() != cols:
        raise KernelError(f"add_rmsnorm_partials: x {tuple(x.shape)} {x.dtype} does not fit the product {tuple(parts.shape)}")
    if cols % 4 or cols > 8192 or (x.data_ptr() | parts.data_ptr() | w.data_ptr()) % 16:
        return add_rmsnorm(x, delta.materialize(), w, eps, add_one)
    out = torch.empty_like(x)
    _check(library().ia_add_rmsnorm_partials(_p(out), _p(x), _p(parts), splits, _p(w), ctypes.c_float(eps), rows, cols,
                                             int(add_one), _stream()))
    return out


def linear(x, w: torch.Tensor, out_dtype: Optional[torch.dtype] = None, mid: bool = True,
           bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x [m, k] . w[n, k]^T (+ bias [n], in the precision of w).  32-bit: `gemm_tiled` (true 32-bit, fixed order).
    bfloat16: the skinny MFMA kernel for up to SKINNY_MAX_ROWS rows, the vendor's GEMM beyond that (the reference uses
    cuBLAS for all of them) or, from 512 rows on where that is faster, gemm_wide.hip (products that `linear_partials` or `gated_linear`
    send there do not come here).
    A 32-bit result of bfloat16 operands (logits) comes straight from the skinny kernel's accumulators for those few
    rows; beyond that it is the vendor's bfloat16 result widened, which is what the reference does for every row (its
    logits are computed in the model's precision and cast for sampling, `inferrs/src/sampler.rs:182`).  From
    `mid_from_rows(k)` rows on (and up to `MID_MAX_ROWS`) a bfloat16 result comes from gemm_mid.hip; `mid=False`: from
    the skinny product or the vendor's GEMM.  The skinny kernel adds a bias to its sums before it rounds them; behind
    every other product a kernel of its own adds it to the stored rows."""
    out_dtype = out_dtype or x.dtype
    if bias is not None and (bias.dtype != w.dtype or bias.numel() != w.shape[0]):
        raise KernelError(f"linear: a bias of {bias.numel()} {bias.dtype} entries for a weight {tuple(w.shape)} {w.dtype}")
    if isinstance(x, NormedRows):
        if _takes_normed_rows(x, w, w.shape[0]):
            _dev(x.scaled, w, x.sums)
            return _stream_product(x.scaled, w, w.shape[0], out_dtype, False, sums_in=x.sums, eps=x.eps, bias=bias)
        x = x.materialize()
    if x.dtype == torch.bfloat16 and skinny_fits(x, w) and x.shape[0] <= SKINNY_MAX_ROWS:
        # (rows that both kernels take: a 32-bit result, the logits head's, stays with the skinny product)
        if out_dtype != torch.bfloat16 or bias is not None or not mid or not mid_fits(x, w):
            return gemm_skinny_bf16(x, w, out_dtype, bias=bias)
    y = _linear_no_bias(x, w, out_dtype if bias is None else x.dtype, mid)
    if bias is None:
        return y
    add_bias(y, bias)
    return widen(y) if out_dtype == torch.float32 and y.dtype != torch.float32 else y


def _linear_no_bias(x: torch.Tensor, w: torch.Tensor, out_dtype: torch.dtype, mid: bool) -> torch.Tensor:
    """The products of `linear` beyond the skinny kernel's rows."""
    if x.dtype == torch.float32:
        return gemm_tiled(x, w, out_dtype)
    m, k = x.shape
    if not skinny_fits(x, w):
        return gemm_tiled(x, w, out_dtype)
    if mid and mid_fits(x, w):
        if out_dtype == torch.float32:
            return gemm_mid_bf16(x, w, torch.float32)
        y = gemm_mid_bf16(x, w, partial=True)
        return y.materialize() if isinstance(y, Partials) else y
    if out_dtype == torch.bfloat16 and _wide_takes("rows", x, w):
        return gemm_wide_rows(x, w)
    _dev(x, w)
    if w.shape[1] != k or w.dtype != x.dtype:
        raise KernelError(f"gemm: x {tuple(x.shape)} {x.dtype} does not fit w {tuple(w.shape)} {w.dtype}")
    if _own_large(x, w):
        y = gemm_mfma_bf16(x, w)
    elif KernelTimer.active is not None:
        y = KernelTimer.active.call("vendor_gemm", vendor_gemm_bf16, x, w)
    else:
        y = vendor_gemm_bf16(x, w)
    return widen(y) if out_dtype == torch.float32 else y


# ---- sampling ---------------------------------------------------------------------------------

def argmax(logits: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The lowest index among each row's maxima, int32 [rows] (into `out` when given)."""
    _dev(logits, out); _f32(logits, "logits")
    rows, vocab = logits.shape
    if out is None:
        out = torch.empty((rows,), dtype=torch.int32, device=logits.device)
    elif out.dtype != torch.int32 or out.numel() != rows:
        raise KernelError(f"argmax: `out` must be int32 [{rows}]")
    words = library().ia_argmax_workspace(rows, vocab)
    ws = torch.empty((words,), dtype=torch.int32, device=logits.device) if words else None
    _check(library().ia_argmax(_p(out), _p(logits), _p(ws), rows, vocab, _stream()))
    return out


def _penalty_args(who: str, rows: int, window: Optional[torch.Tensor], repetition: Optional[torch.Tensor],
                  frequency: Optional[torch.Tensor], presence: Optional[torch.Tensor], bias_ids: Optional[torch.Tensor] = None,
                  bias_vals: Optional[torch.Tensor] = None) -> tuple:
    """Bias and penalties of `rows` rows, checked, as the entry points take them."""
    _dev(window, repetition, frequency, presence, bias_ids, bias_vals)
    _f32(repetition, "repetition"); _f32(frequency, "frequency"); _f32(presence, "presence")
    w = 0 if window is None else window.shape[1]
    nb = 0 if bias_ids is None else bias_ids.shape[1]
    if window is not None:
        _i32(window, "window")
        if window.shape[0] != rows:
            raise KernelError(f"{who}: one window row per row of logits")
    if (bias_ids is None) != (bias_vals is None):
        raise KernelError(f"{who}: bias ids and values come together")
    if bias_ids is not None:
        _i32(bias_ids, "bias_ids"); _f32(bias_vals, "bias_vals")
        if bias_ids.shape != bias_vals.shape or bias_ids.shape[0] != rows:
            raise KernelError(f"{who}: bias arrays must be [rows, entries]")
    for t in (repetition, frequency, presence):
        if t.numel() != rows:
            raise KernelError(f"{who}: one penalty value per row of logits")
    return _p(window), w, _p(repetition), _p(frequency), _p(presence), _p(bias_ids), _p(bias_vals), nb


def penalize(logits: torch.Tensor, window: Optional[torch.Tensor], repetition: torch.Tensor,
             frequency: torch.Tensor, presence: torch.Tensor, bias_ids: Optional[torch.Tensor] = None,
             bias_vals: Optional[torch.Tensor] = None) -> torch.Tensor:
    """In place on float32 logits [rows, vocab]: logit bias, then repetition, frequency and presence
    penalties over each row's `window` of earlier tokens (int32 [rows, w], -1 = none)."""
    _dev(logits)
    _f32(logits, "logits")
    rows, vocab = logits.shape
    args = _penalty_args("penalize", rows, window, repetition, frequency, presence, bias_ids, bias_vals)
    _check(library().ia_penalize(_p(logits), rows, vocab, *args, _stream()))
    return logits


def window_push(window: torch.Tensor, caps: torch.Tensor, tokens: torch.Tensor) -> torch.Tensor:
    """In place: every row's penalty window [rows, w] (int32, -1 = empty) takes the row's new token; row i
    keeps its last caps[i] tokens (0: no window)."""
    _dev(window, caps, tokens)
    _i32(window, "window"); _i32(caps, "caps"); _i32(tokens, "tokens")
    rows, w = window.shape
    if caps.numel() != rows or tokens.numel() != rows or not window.is_contiguous():
        raise KernelError("window_push: one cap and one token per row of a contiguous window")
    _check(library().ia_window_push(_p(window), rows, w, _p(caps), _p(tokens), _stream()))
    return window


_NO_PENALTIES = (None, 0, None, None, None, None, None, 0)


def sample_narrow_top() -> int:
    """Rows with a top_k of up to this many, below the vocabulary, are drawn from a few candidates of every stretch of the row,
    but for those that `sample_is_narrow` leaves out."""
    return library().ia_sample_narrow_top()


def sample_is_narrow(top_k: int, vocab: int, temperature: float, top_p: float, min_p: float, n_top: int = -1,
                     biased: bool = False) -> bool:
    """Whether `sample` draws a row with these parameters from a few candidates of every stretch (`narrow_only`): a top_k in 1 ..
    `sample_narrow_top()`, unless the row reports two entries and more of a list that neither top_p nor min_p ends, at a low
    temperature or with a logit bias: those entries lie beyond the candidates."""
    return bool(library().ia_sample_is_narrow(top_k, vocab, ctypes.c_float(temperature), ctypes.c_float(top_p),
                                              ctypes.c_float(min_p), n_top, int(biased)))


def sample(logits: torch.Tensor, temperature: torch.Tensor, top_k: torch.Tensor, top_p: torch.Tensor,
           min_p: torch.Tensor, u: torch.Tensor, n_top: Optional[torch.Tensor] = None, *,
           penalties: Optional[tuple] = None, narrow_only: bool = False, out: Optional[torch.Tensor] = None):
    """One token per row of float32 logits: greedy where temperature < 1e-5, else temperature,
    top-k, top-p, min-p and the walk to the row's random number u in [0, 1).  With `n_top` (int32
    per row: -1 none, else 0..20) also returns the log-probabilities within the kept list, float32
    [rows, 1 + 20] (the drawn token's, then the list's first entries'), and those entries' ids, int32
    [rows, 20] (-1: no entry): the result is then (tokens, log-probabilities, ids).
    `penalties`: what `penalize` takes behind the logits, applied on the way (the logits stay as they are).
    `narrow_only`: the caller knows that every row is greedy or one that `sample_is_narrow`, and saves a launch.  `out`: where the tokens go (int32 [rows])."""
    _dev(logits, temperature, top_k, top_p, min_p, u, n_top, out)
    _f32(logits, "logits"); _f32(temperature, "temperature"); _f32(top_p, "top_p"); _f32(min_p, "min_p"); _f32(u, "u")
    _i32(top_k, "top_k")
    rows, vocab = logits.shape
    for t in (temperature, top_k, top_p, min_p, u) + ((n_top,) if n_top is not None else ()):
        if t.numel() != rows:
            raise KernelError("sample: one parameter value per row of logits")
    pen = _NO_PENALTIES if penalties is None else _penalty_args("sample", rows, *penalties)
    lib = library()
    if out is None:
        out = torch.empty((rows,), dtype=torch.int32, device=logits.device)
    else:
        _i32(out, "out")
        if out.numel() != rows:
            raise KernelError("sample: one place per row of logits")
    ws = torch.empty((lib.ia_sample_workspace(rows, vocab),), dtype=torch.int32, device=logits.device)
    lp = ids = None
    if n_top is not None:
        _i32(n_top, "n_top")
        most = lib.ia_sample_max_top()
        lp = torch.empty((rows, 1 + most), dtype=torch.float32, device=logits.device)
        ids = torch.empty((rows, most), dtype=torch.int32, device=logits.device)
    _check(lib.ia_sample(_p(out), _p(logits), _p(ws), rows, vocab, _p(temperature), _p(top_k), _p(top_p),
                         _p(min_p), _p(u), _p(n_top), _p(lp), _p(ids), *pen, int(narrow_only), _stream()))
    return out if n_top is None else (out, lp, ids)


def sample_packed(logits: torch.Tensor, words: torch.Tensor, width: int, n_bias: int, *, penalized: bool,
                  narrow_only: bool) -> torch.Tensor:
    """`sample` of rows whose parameters lie one behind another in `words` (32-bit words on the device; an array a parameter, a row's
    entries together): with `penalized` the windows [rows, width] (none for a width of 0), the repetition, frequency and presence
    penalties, the biases' ids and values [rows, n_bias]; then temperature, top_k, top_p, min_p and u."""
    _dev(logits, words); _f32(logits, "logits"); _i32(words, "words")
    rows, vocab = logits.shape
    if words.numel() < rows * ((width + 3 + 2 * n_bias if penalized else 0) + 5):
        raise KernelError(f"sample_packed: {words.numel()} words for {rows} rows, windows of {width} and {n_bias} biases")
    at, step = _p(words), 4 * rows
    pen = _NO_PENALTIES
    if penalized:
        rep = at + width * step
        ids = rep + 3 * step
        pen = (at if width else None, width, rep, rep + step, rep + 2 * step, ids if n_bias else None,
               ids + n_bias * step if n_bias else None, n_bias)
        at = ids + 2 * n_bias * step
    out = torch.empty((rows,), dtype=torch.int32, device=logits.device)
    ws = torch.empty((_sample_workspace(rows, vocab),), dtype=torch.int32, device=logits.device)
    _check(library().ia_sample(_p(out), _p(logits), _p(ws), rows, vocab, at, at + step, at + 2 * step, at + 3 * step, at + 4 * step,
                               None, None, None, *pen, int(narrow_only), _stream()))
    return out


@functools.lru_cache(maxsize=256)
def _sample_workspace(rows: int, vocab: int) -> int:
    return _raw_library().ia_sample_workspace(rows, vocab)


def _mid_dual_fits(x: torch.Tensor, w_gate_up: torch.Tensor) -> bool:
    """[gate; up] at up to 16 rows on gemm_mid.hip: where the weight makes a block for every compute unit."""
    return (w_gate_up.shape[0] % 2 == 0 and mid_fits(x, w_gate_up, few_rows=True)
            and w_gate_up.numel() * w_gate_up.element_size() <= MID_DUAL_MAX_BYTES
            and bool(library().ia_gemm_mid_fills(w_gate_up.shape[0] // 2, w_gate_up.shape[1], 1)))


def gated_linear(x, w_gate_up: torch.Tensor, activation: str = "silu",
                 bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """act(x . gate^T) * (x . up^T) for w_gate_up = [gate; up] (`activation`: a name of `ACTIVATIONS`; `bias`
    [2 n]: added to both products before the activation): one fused kernel for few bfloat16 rows, else the
    product followed by the element-wise kernel."""
    # (few rows too go to gemm_mid.hip where its blocks fill the chip evenly: inside a decode step the pair of this product
    # and the next takes 58.0 us against 60.6 at 8 rows and 60.4 against 67.2 at 16, sizes of an 8B model)
    activation_code(activation)
    even = w_gate_up.shape[0] % 2 == 0
    if isinstance(x, NormedRows):
        if even and _takes_normed_rows(x, w_gate_up, w_gate_up.shape[0] // 2):
            _dev(x.scaled, w_gate_up, x.sums)
            if bias is None and _mid_dual_fits(x.scaled, w_gate_up):
                return gemm_mid_bf16(x.scaled, w_gate_up, dual=True, sums_in=x.sums, eps=x.eps, activation=activation)
            return _stream_product(x.scaled, w_gate_up, w_gate_up.shape[0] // 2, x.scaled.dtype, True,
                                   sums_in=x.sums, eps=x.eps, activation=activation, bias=bias)
        x = x.materialize()
    if x.shape[0] <= SKINNY_MAX_ROWS and skinny_fits(x, w_gate_up):
        if bias is None and (_mid_dual_fits(x, w_gate_up) or (
                even and mid_fits(x, w_gate_up) and w_gate_up.numel() * w_gate_up.element_size() <= MID_DUAL_MAX_BYTES)):
            return gemm_mid_bf16(x, w_gate_up, dual=True, activation=activation)
        return gemm_skinny_bf16(x, w_gate_up, x.dtype, dual=True, activation=activation, bias=bias)
    if bias is None:
        if (even and mid_fits(x, w_gate_up)
                and w_gate_up.numel() * w_gate_up.element_size() <= MID_DUAL_MAX_BYTES):
            return gemm_mid_bf16(x, w_gate_up, dual=True, activation=activation)
        if (x.shape[0] > MID_MAX_ROWS and w_gate_up.shape[0] % 8 == 0
                and any(_wide_pays(rule, x.shape[0], w_gate_up.shape[0] // 2, x.shape[1]) for rule in ("dual", "narrow"))
                and wide_fits(x, w_gate_up)):
            return gemm_wide_bf16(x, w_gate_up, dual=True, activation=activation)
        if even and x.dtype == torch.bfloat16 and skinny_fits(x, w_gate_up) and _own_large(x, w_gate_up):
            return gemm_mfma_bf16(x, w_gate_up, dual=True, activation=activation)
    # (a [gate; up] beyond MID_DUAL_MAX_BYTES at 17 to 64 rows: the vendor's GEMM, not the plain product of gemm_mid.hip)
    return gate_mul(linear(x, w_gate_up, mid=bias is not None, bias=bias), activation)


def gated_silu_linear(x, w_gate_up: torch.Tensor) -> torch.Tensor:
    """`gated_linear` with SiLU and no bias."""
    return gated_linear(x, w_gate_up, "silu")


# ---- several residual streams, latent attention, gated recurrence, routed experts -----------------
from .mix import (clamped_gate_mul, conv_step, embed_gather_scaled, experts_forward, gate_rows, head_product,    # noqa: E402
                  latent_prep, norm_slice, parallel_step, postnorm_step, rglru_scan, route, scale_inplace, sigmoid_gate, softcap,
                  streams_open, streams_step)
from .state import (activation, conv_act_step, exp_gates, group_norm_gate, linear_scan, sandwich_step,   # noqa: E402
                    step_gates)
from . import state                                                                                    # noqa: E402
from .gated import branch_step, conv_qkv, differ_norm, fading_scan                                     # noqa: E402
from . import gated                                                                                    # noqa: E402
