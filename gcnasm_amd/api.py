"""ctypes front end of the C ABI declared in include/mi355_a8w8.h.

Argument names and meanings follow struct opus_gemm_kargs of the reference
(opus_gemm/block_scale_gemm/gemm_a8w8_blockscale_common.h:4-25): element strides, A [M,K]
and B [N,K] row-major E4M3 bytes, C [M,N].  Tensors are torch tensors used purely as
device-memory handles (data_ptr) plus the current HIP stream.
"""
import ctypes
import os
import subprocess
import warnings

_HERE = os.path.dirname(os.path.abspath(__file__))
# MI355_A8W8_LIBRARY: another build of the same sources (a measurement build made with `make EXTRA=-D... OUT=...`),
# for A/B timings of one program against two libraries; unset, the library next to this file
_SO = os.environ.get("MI355_A8W8_LIBRARY") or os.path.join(_HERE, "libmi355a8w8.so")

TENSOR, ROWCOL, BLOCK, MX, MX_TILED = 0, 1, 2, 3, 4
BF16, FP32 = 0, 1
OCP, FNUZ = 0, 1


class A8W8Error(RuntimeError):
    def __init__(self, status, where):
        self.status = status
        super().__init__(f"{where}: {status_string(status)} (status {status})")


class WeightHeader(ctypes.Structure):
    _fields_ = [("magic", ctypes.c_char * 8), ("version", ctypes.c_uint32), ("n", ctypes.c_uint32), ("k", ctypes.c_uint32),
                ("b_preshuffled", ctypes.c_uint32), ("scale_mode", ctypes.c_uint32), ("reserved", ctypes.c_uint32),
                ("b_bytes", ctypes.c_uint64), ("scale_bytes", ctypes.c_uint64), ("checksum", ctypes.c_uint64),
                ("reserved2", ctypes.c_uint64)]


class GemmArgs(ctypes.Structure):
    _fields_ = [
        ("a", ctypes.c_void_p), ("b", ctypes.c_void_p), ("c", ctypes.c_void_p),
        ("m", ctypes.c_int), ("n", ctypes.c_int), ("k", ctypes.c_int), ("batch", ctypes.c_int),
        ("stride_a", ctypes.c_int), ("stride_b", ctypes.c_int), ("stride_c", ctypes.c_int),
        ("stride_a_batch", ctypes.c_int), ("stride_b_batch", ctypes.c_int), ("stride_c_batch", ctypes.c_int),
        ("sfa", ctypes.c_void_p), ("sfb", ctypes.c_void_p),
        ("stride_sfa", ctypes.c_int), ("stride_sfb", ctypes.c_int),
        ("stride_sfa_batch", ctypes.c_int), ("stride_sfb_batch", ctypes.c_int),
        ("scale_mode", ctypes.c_int), ("c_dtype", ctypes.c_int), ("b_preshuffled", ctypes.c_int),
    ]


def library_path():
    return _SO


def build_library(verbose=False):
    """Compile the HIP sources for gfx950 with hipcc (cross-compiles without a GPU) and the host's binding."""
    subprocess.check_call(["make", "-C", os.path.join(_HERE, "csrc"), "-B"],
                          stdout=None if verbose else subprocess.DEVNULL,
                          stderr=None if verbose else subprocess.DEVNULL)
    return _SO


_lib = None
torch = None        # imported with the first call that takes tensors (the package itself needs only ctypes)


def _need_torch():
    global torch
    if torch is None:
        import torch as module
        torch = module


def lib():
    """The loaded C ABI.  Raises if the library has not been built; never substitutes a CPU path."""
    global _lib
    if _lib is None:
        if not os.path.exists(_SO):
            raise FileNotFoundError(
                f"{_SO} is missing: build it with gcnasm_amd.build_library() or `make -C gcnasm_amd/csrc`")
        L = ctypes.CDLL(_SO)
        vp = ctypes.c_void_p
        L.a8w8_gemm.argtypes = [ctypes.POINTER(GemmArgs), vp]
        L.a8w8_gemm_blockscale.argtypes = [ctypes.POINTER(GemmArgs), vp]
        L.a16w16_gemm.argtypes = [ctypes.POINTER(GemmArgs), vp]
        L.a16w16_flatmm.argtypes = [ctypes.POINTER(GemmArgs), vp]
        L.a4w4_gemm.argtypes = [ctypes.POINTER(GemmArgs), vp]
        L.a4w4_flatmm.argtypes = [ctypes.POINTER(GemmArgs), vp]
        L.a4w4_quantize_mx.argtypes = [vp, ctypes.c_int, ctypes.c_int, ctypes.c_int, vp, vp, ctypes.c_int, vp]
        L.a8w8_flatmm.argtypes = [ctypes.POINTER(GemmArgs), vp]
        L.a8w8_preshuffle_b.argtypes = [vp, vp, ctypes.c_int, ctypes.c_int]
        L.a8w8_unshuffle_b.argtypes = [vp, vp, ctypes.c_int, ctypes.c_int]
        L.a8w8_preshuffle_b_device.argtypes = [vp, vp, ctypes.c_int, ctypes.c_int, vp]
        L.a8w8_cvt_f32_to_e4m3.argtypes = [vp, vp, ctypes.c_size_t, ctypes.c_int, ctypes.c_int, vp]
        L.a8w8_cvt_e4m3_to_f32.argtypes = [vp, vp, ctypes.c_size_t, ctypes.c_int, vp]
        L.a8w8_quantize.argtypes = [vp, ctypes.c_int, ctypes.c_int, ctypes.c_int, vp, vp, ctypes.c_int,
                                    ctypes.c_int, vp]
        if hasattr(L, "a8w8_quantize_ws"):      # (not in an older build named by MI355_A8W8_LIBRARY)
            L.a8w8_quantize_ws.argtypes = [vp, ctypes.c_int, ctypes.c_int, ctypes.c_int, vp, vp, ctypes.c_int, ctypes.c_int, vp, ctypes.c_size_t, vp]
            L.a8w8_quantize_workspace_bytes.restype = ctypes.c_size_t
            L.a8w8_quantize_workspace_bytes.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int]
        L.a8w8_mx_tile_scales.argtypes = [vp, ctypes.c_int, ctypes.c_int, ctypes.c_int, vp, vp]
        L.a8w8_mx_tile_scales_ab.argtypes = [vp, ctypes.c_int, ctypes.c_int, vp, vp, ctypes.c_int, ctypes.c_int, vp,
                                             ctypes.c_int, vp]
        L.a8w8_mx_tiled_bytes.restype = ctypes.c_size_t
        L.a8w8_mx_tiled_bytes.argtypes = [ctypes.c_int, ctypes.c_int]
        L.a8w8_weight_scale_bytes.restype = ctypes.c_size_t
        L.a8w8_weight_scale_bytes.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int]
        L.a8w8_weights_save.argtypes = [ctypes.c_char_p, vp, vp, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int]
        L.a8w8_weights_info.argtypes = [ctypes.c_char_p, ctypes.POINTER(WeightHeader)]
        L.a8w8_weights_load.argtypes = [ctypes.c_char_p, vp, ctypes.c_size_t, vp, ctypes.c_size_t]
        L.a8w8_status_string.restype = ctypes.c_char_p
        L.a8w8_status_string.argtypes = [ctypes.c_int]
        L.a8w8_kernel_name.restype = ctypes.c_char_p
        L.a8w8_kernel_name.argtypes = [ctypes.POINTER(GemmArgs)]
        L.a8w8_version.restype = ctypes.c_int
        L.a8w8_init.argtypes = [ctypes.c_int]
        L.a8w8_hbm_read_probe.argtypes = [vp, ctypes.c_size_t, vp, vp]
        L.a8w8_route_override.argtypes = [ctypes.c_int]
        _lib = L
    return _lib


def status_string(status):
    return lib().a8w8_status_string(int(status)).decode()


# The host's part of a call is what a decoding step of a small layer waits for (1 x 4096 x 4096 with its quantiser: the two
# launches take 8 us of device time).  Hence the compiled path (csrc/binding.cpp) for ordinary tensors: the functions below try it first, and
# go through their own statements where it answers None -- to name what is wrong with the arguments, or for tensor subclasses and active modes.
_OPS = ("a8w8_gemm", "a8w8_gemm_blockscale", "a8w8_flatmm", "a16w16_gemm", "a16w16_flatmm", "a4w4_gemm", "a4w4_flatmm")
_GEMM, _BLOCKSCALE, _FLATMM, _GEMM16, _FLATMM16, _GEMM4, _FLATMM4 = range(7)


def _torch_build():
    """What the Makefile compiles into the module as torch_build."""
    return f"{torch.__version__} {torch.version.git_version}"


def _connect():
    """Load csrc/binding.cpp's module on the first call that takes tensors and hand it the library's entry points.  Without a module for this torch, or with
    a library older than the module, the functions' own statements serve every call: the same kernels, 4 to 8 us of host time more per call."""
    global _fast_gemm, _fast_quantize, _fast_quantize_mxfp4, _fast_encode, _fast_decode
    _need_torch()
    L = lib()
    why = None
    try:
        from . import _binding
        if _binding.torch_build != _torch_build():
            why = f"it was built for torch {_binding.torch_build}, this is {_torch_build()}"
        elif not hasattr(L, "a8w8_quantize_ws"):
            why = f"{_SO} has no a8w8_quantize_ws"
    except ImportError as e:
        why = str(e)
    if why is not None:
        warnings.warn(f"{os.path.join(_HERE, '_binding.so')} is not used: {why}.  Calls take longer on the host; build it with gcnasm_amd.build_library() or "
                      "`make -C gcnasm_amd/csrc`.", RuntimeWarning, stacklevel=4)
        _fast_gemm = _fast_quantize = _fast_quantize_mxfp4 = _fast_encode = _fast_decode = lambda *args: None
        return
    _binding.connect(*(ctypes.cast(getattr(L, f), ctypes.c_void_p).value
                       for f in _OPS + ("a8w8_quantize_ws", "a4w4_quantize_mx", "a8w8_cvt_f32_to_e4m3", "a8w8_cvt_e4m3_to_f32",
                                        "a8w8_quantize_workspace_bytes")))
    _fast_gemm, _fast_quantize, _fast_quantize_mxfp4 = _binding.gemm, _binding.quantize, _binding.quantize_mxfp4
    _fast_encode, _fast_decode = _binding.encode, _binding.decode


def _fast_gemm(*args):
    _connect()
    return _fast_gemm(*args)


def _fast_quantize(*args):
    _connect()
    return _fast_quantize(*args)


def _fast_quantize_mxfp4(*args):
    _connect()
    return _fast_quantize_mxfp4(*args)


def _fast_encode(*args):
    _connect()
    return _fast_encode(*args)


def _fast_decode(*args):
    _connect()
    return _fast_decode(*args)


def _done(result, where):
    """What the compiled path returned: the outputs, or the status of a call that the library refused."""
    if type(result) is int:
        raise A8W8Error(result, where)
    return result


def _stream():
    """The current stream's handle (what torch.cuda.current_stream().cuda_stream holds, without the object around it)."""
    _need_torch()
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def _check(status, where):
    if status != 0:
        raise A8W8Error(status, where)


def raw_gemm_args(a, b, c, sfa, sfb, m, n, k, scale_mode, c_dtype=BF16, batch=1, stride_a=None, stride_b=None,
                  stride_c=None, stride_sfa=None, stride_sfb=None, b_preshuffled=0, batch_strides=None):
    """Fill the C argument block from raw integers (device addresses)."""
    if stride_a is None:
        stride_a = k
    if stride_b is None:
        stride_b = k
    if stride_c is None:
        stride_c = n
    if stride_sfa is None:
        stride_sfa = m if scale_mode == BLOCK else k // 32 if scale_mode == MX else 0
    if stride_sfb is None:
        stride_sfb = 1 if scale_mode == ROWCOL else k // 128 if scale_mode == BLOCK else k // 32 if scale_mode == MX else 0
    if batch_strides is not None:
        a_b, b_b, c_b, sfa_b, sfb_b = batch_strides
    else:
        a_b, b_b, c_b = m * stride_a, n * stride_b, m * stride_c
        if scale_mode == TENSOR:
            sfa_b = sfb_b = 1
        elif scale_mode == ROWCOL:
            sfa_b, sfb_b = m, n
        elif scale_mode == BLOCK:
            sfa_b, sfb_b = m * (k // 128), (n // 128) * (k // 128)
        elif scale_mode == MX:
            sfa_b, sfb_b = m * (k // 32), n * (k // 32)
        elif scale_mode == MX_TILED:
            sfa_b, sfb_b = mx_tiled_bytes(m, k), mx_tiled_bytes(n, k)
        else:
            sfa_b = sfb_b = 0
    # (in the order of the fields)
    return GemmArgs(a, b, c, m, n, k, batch, stride_a, stride_b, stride_c, a_b, b_b, c_b, sfa, sfb, stride_sfa, stride_sfb, sfa_b, sfb_b,
                    scale_mode, c_dtype, b_preshuffled)


def mx_tiled_bytes(rows, k):
    """Size of one matrix's E8M0 scales in the MX_TILED layout."""
    return ((k + 511) // 512) * ((rows + 63) // 64) * 1024


def _out(c, shape, c_dtype, device):
    """The output tensor and its C type code: a caller's tensor decides the type (bf16 or fp32 only)."""
    if c is None:
        return torch.empty(shape, dtype=torch.bfloat16 if c_dtype == BF16 else torch.float32, device=device), c_dtype
    if c.dtype not in (torch.bfloat16, torch.float32):
        raise TypeError(f"output tensor must be bfloat16 or float32, got {c.dtype}")
    if tuple(c.shape) != tuple(shape):
        raise ValueError(f"output tensor has shape {tuple(c.shape)}, expected {tuple(shape)}")
    if shape[-1] > 1 and c.stride(-1) != 1:
        raise ValueError("c: the last dimension must be contiguous")
    if not c.is_cuda:
        raise ValueError("c must live on the GPU")
    return c, (BF16 if c.dtype == torch.bfloat16 else FP32)


def _check_rows(t, name, element_bytes):
    """What is read row by row: elements of the size that the kernel takes, side by side in GPU memory.  Anything else would be misread, and smaller
    elements read past their end."""
    if t.element_size() != element_bytes:
        raise TypeError(f"{name} must have elements of {element_bytes} bytes, got {t.dtype}")
    if t.shape[-1] > 1 and t.stride(-1) != 1:
        raise ValueError(f"{name}: the last dimension must be contiguous (stride {t.stride(-1)})")
    if not t.is_cuda:
        raise ValueError(f"{name} must live on the GPU")


def _check_ints(where, *values):
    """The C ABI counts rows, columns and strides with an int; a larger one would be read modulo 2^32."""
    if any(v > 0x7FFFFFFF for v in values):
        raise A8W8Error(-7, where)


def _check_fp32_rows(x, where):
    if x.dtype != torch.float32:
        raise TypeError(f"x must be float32, got {x.dtype}")
    _check_rows(x, "x", 4)
    _check_ints(where, x.shape[0], x.shape[1], x.stride(0))


def _check_operands(a, b, element_bytes, dims, n=None):
    """a [.., M, row], and b [.., N, row] or, with `n` given, the flat pre-shuffled weight of n rows (any element type)."""
    for t, name, want in ((a, "a", dims), (b, "b", dims if n is None else (1, 2))):
        if t.dim() not in want:
            raise ValueError(f"{name} must have {' or '.join(str(d) for d in want)} dimensions, got {t.dim()}")
    _check_rows(a, "a", element_bytes)
    if n is None:
        _check_rows(b, "b", element_bytes)
        if b.shape[-1] < a.shape[-1]:
            raise ValueError(f"rows of b hold {b.shape[-1]} elements, those of a {a.shape[-1]}")
        return
    if not b.is_contiguous() or not b.is_cuda:
        raise ValueError("shuffled b must be a contiguous GPU tensor")
    if b.numel() * b.element_size() < n * a.shape[-1] * element_bytes:
        raise ValueError(f"shuffled b holds {b.numel() * b.element_size()} bytes, {n} rows are {n * a.shape[-1] * element_bytes}")


def _check_scales(t, name, scale_mode):
    """Scale arrays are read with the strides their shape implies: they have to be contiguous, on the GPU, and of
    the element type of the scale mode (fp32, or uint8 for the E8M0 modes)."""
    want = torch.uint8 if scale_mode in (MX, MX_TILED) else torch.float32
    if not t.is_cuda or not t.is_contiguous():
        raise ValueError(f"{name} must be a contiguous GPU tensor")
    if t.dtype != want:
        raise TypeError(f"{name} must be {want} for this scale mode, got {t.dtype}")


def scale_elements(scale_mode, rows, k, weight_side):
    """Elements one batch entry's scale array holds for a matrix of `rows` rows (A: weight_side False, B: True), as the
    kernels index it with the default strides of raw_gemm_args."""
    if scale_mode == TENSOR:
        return 1
    if scale_mode == ROWCOL:
        return rows
    if scale_mode == BLOCK:
        return ((rows + 127) // 128 if weight_side else rows) * (k // 128)
    if scale_mode == MX:
        return rows * (k // 32)
    return mx_tiled_bytes(rows, k)


def _check_scale_sizes(sfa, sfb, scale_mode, m, n, k, batch, b_shared):
    """An undersized scale array would be read past its end on the device; weights shared by all batch entries come with
    one set of weight scales (a per-entry set would silently be used for entry 0 only)."""
    need_a = batch * scale_elements(scale_mode, m, k, False)
    per_b = scale_elements(scale_mode, n, k, True)
    need_b = per_b if b_shared else batch * per_b
    has_a, has_b = sfa.numel(), sfb.numel()
    if has_a < need_a:
        raise ValueError(f"sfa holds {has_a} elements, this problem reads {need_a}")
    if has_b < need_b:
        raise ValueError(f"sfb holds {has_b} elements, this problem reads {need_b}")
    if b_shared and has_b >= batch * per_b and has_b > per_b:
        raise ValueError(f"b is shared by all {batch} batch entries but sfb holds a set of scales per entry; pass one set")


def _check_fp4_scales(sfa, sfb, scale_mode, m, n, k):
    """E8M0 bytes of any one-byte type, contiguous, on the GPU, as many as the kernels read (the library refuses other modes)."""
    if scale_mode not in (MX, MX_TILED):
        return
    for t, name, rows in ((sfa, "sfa", m), (sfb, "sfb", n)):
        if t.element_size() != 1:
            raise TypeError(f"{name} must have elements of one byte, got {t.dtype}")
        if not t.is_contiguous() or not t.is_cuda:
            raise ValueError(f"{name} must be a contiguous GPU tensor")
        need = scale_elements(scale_mode, rows, k, name == "sfb")
        if t.numel() < need:
            raise ValueError(f"{name} holds {t.numel()} elements, this problem reads {need}")


def _args_from_tensors(a, b, sfa, sfb, scale_mode, c, c_dtype, b_preshuffled, n=None, scaled=True):
    _need_torch()
    a_shape, a_strides, b_shape, b_strides = a.shape, a.stride(), b.shape, b.stride()
    if b_preshuffled and n is None:
        n = b_shape[-2]
    _check_operands(a, b, 1 if scaled else 2, (2, 3), n=n if b_preshuffled else None)
    if scaled:
        _check_scales(sfa, "sfa", scale_mode)
        _check_scales(sfb, "sfb", scale_mode)
    batched = len(a_shape) == 3
    batch = a_shape[0] if batched else 1
    m, k = a_shape[-2], a_shape[-1]
    if n is None:
        n = b_shape[-2]
    c, c_dtype = _out(c, (batch, m, n) if batched else (m, n), c_dtype, a.device)
    c_strides = c.stride()
    _check_ints("gemm", m, n, k, batch, a_strides[-2], k if b_preshuffled else b_strides[-2], c_strides[-2])
    if batch > 1:
        _check_ints("gemm", a_strides[0], b_strides[0] if len(b_shape) == 3 else n * k if b_preshuffled else 0, c_strides[0])
    g = raw_gemm_args(a.data_ptr(), b.data_ptr(), c.data_ptr(), sfa.data_ptr(), sfb.data_ptr(), m, n, k, scale_mode,
                      c_dtype, batch, stride_a=a_strides[-2], stride_b=(k if b_preshuffled else b_strides[-2]),
                      stride_c=c_strides[-2], b_preshuffled=b_preshuffled)
    if batched:
        g.stride_a_batch, g.stride_c_batch = a_strides[0], c_strides[0]
        if b_preshuffled:
            # flat shuffled weights: of every batch entry back to back, or one matrix shared by all of them
            per_entry = n * k * a.element_size() // b.element_size()
            if b.numel() == batch * per_entry:
                g.stride_b_batch = n * k
            elif b.numel() == per_entry:
                g.stride_b_batch = 0
                g.stride_sfb_batch = 0
            else:
                raise ValueError(f"shuffled b holds {b.numel()} elements, expected {per_entry} or {batch} x {per_entry}")
        elif len(b_shape) == 3:
            if b_shape[0] != batch:
                raise ValueError(f"b has {b_shape[0]} batch entries, a has {batch}")
            g.stride_b_batch = b_strides[0]
        else:
            # one weight matrix shared by every batch entry, and with it one set of weight scales
            g.stride_b_batch = 0
            g.stride_sfb_batch = 0
    if scaled:
        _check_scale_sizes(sfa, sfb, scale_mode, m, n, k, batch, b_shared=(batch > 1 and g.stride_b_batch == 0))
    return g, c


def gemm(a, b, sfa, sfb, scale_mode, c=None, c_dtype=BF16, n=None):
    """C = dequant(A) @ dequant(B)^T through a8w8_gemm.  a [.., M, K] u8, b [.., N, K] u8 on the GPU; with `n` given,
    b is the flat pre-shuffled weight (preshuffle_b_device) of n rows."""
    r = _fast_gemm(_GEMM, a, b, sfa, sfb, scale_mode, c, c_dtype, n)
    if r is not None:
        return _done(r, "a8w8_gemm")
    g, c = _args_from_tensors(a, b, sfa, sfb, scale_mode, c, c_dtype, 0 if n is None else 1, n=n)
    _check(lib().a8w8_gemm(ctypes.byref(g), _stream()), "a8w8_gemm")
    return c


def gemm_a16w16(a, b, c=None, c_dtype=BF16, n=None):
    """C = A @ B^T for bf16 a [.., M, K] and b [.., N, K] (torch.bfloat16 on the GPU) through a16w16_gemm; with `n`
    given, b is the flat pre-shuffled weight of n rows (preshuffle_b_bf16_device)."""
    r = _fast_gemm(_GEMM16, a, b, a, b, TENSOR, c, c_dtype, n)
    if r is not None:
        return _done(r, "a16w16_gemm")
    g, c = _args_from_tensors(a, b, a, b, TENSOR, c, c_dtype, 0 if n is None else 1, n=n, scaled=False)
    _check(lib().a16w16_gemm(ctypes.byref(g), _stream()), "a16w16_gemm")
    return c


def preshuffle_b_bf16_device(b):
    """bf16 weights [N, K] on the GPU -> the pre-shuffled byte layout a16w16_flatmm streams (flat uint8 tensor)."""
    _need_torch()
    n, k = b.shape
    return preshuffle_b_device(b.contiguous().view(torch.uint8).view(n, 2 * k))


def flatmm_a16w16(a, b_shuffled, n, c=None, c_dtype=BF16):
    """Skinny-M bf16 GEMM over weights from preshuffle_b_bf16_device."""
    r = None if n is None else _fast_gemm(_FLATMM16, a, b_shuffled, a, a, TENSOR, c, c_dtype, n)
    if r is not None:
        return _done(r, "a16w16_flatmm")
    g, c = _args_from_tensors(a, b_shuffled, a, a, TENSOR, c, c_dtype, 1, n=n, scaled=False)
    _check(lib().a16w16_flatmm(ctypes.byref(g), _stream()), "a16w16_flatmm")
    return c


def quantize_mxfp4(x, tiled=False):
    """fp32 [rows, K] -> (packed E2M1 bytes [rows, K/2], E8M0 scales row-major [rows, K/32] or tiled)."""
    r = _fast_quantize_mxfp4(x, tiled)
    if r is not None:
        return _done(r, "a4w4_quantize_mx")
    _need_torch()
    rows, k = x.shape
    _check_fp32_rows(x, "a4w4_quantize_mx")
    q = torch.empty((rows, k // 2), dtype=torch.uint8, device=x.device)
    s = torch.empty(mx_tiled_bytes(rows, k) if tiled else (rows, k // 32), dtype=torch.uint8, device=x.device)
    _check(lib().a4w4_quantize_mx(x.data_ptr(), rows, k, x.stride(0), q.data_ptr(), s.data_ptr(), int(tiled), _stream()),
           "a4w4_quantize_mx")
    return q, s


def gemm_a4w4(a, b, sfa, sfb, scale_mode=MX_TILED, c=None, c_dtype=BF16, n=None):
    """MXFP4 GEMM through a4w4_gemm: a [M, K/2], b [N, K/2] packed E2M1 (uint8 on the GPU); with `n` given, b is the
    flat pre-shuffled weight of n rows (preshuffle_b_device on the packed bytes)."""
    r = _fast_gemm(_GEMM4, a, b, sfa, sfb, scale_mode, c, c_dtype, n)
    if r is not None:
        return _done(r, "a4w4_gemm")
    _need_torch()
    _check_operands(a, b, 1, (2,), n=n)
    m, k = a.shape[-2], a.shape[-1] * 2
    shuffled = n is not None
    if not shuffled:
        n = b.shape[-2]
    _check_fp4_scales(sfa, sfb, scale_mode, m, n, k)
    c, c_dtype = _out(c, (m, n), c_dtype, a.device)
    _check_ints("a4w4_gemm", m, n, k, 2 * a.stride(-2), k if shuffled else 2 * b.stride(-2), c.stride(-2))
    g = raw_gemm_args(a.data_ptr(), b.data_ptr(), c.data_ptr(), sfa.data_ptr(), sfb.data_ptr(), m, n, k, scale_mode, c_dtype,
                      stride_a=a.stride(-2) * 2, stride_b=(k if shuffled else b.stride(-2) * 2), stride_c=c.stride(-2),
                      b_preshuffled=int(shuffled))
    _check(lib().a4w4_gemm(ctypes.byref(g), _stream()), "a4w4_gemm")
    return c


def flatmm_a4w4(a, b_shuffled, sfa_tiled, sfb_tiled, n, c=None, c_dtype=BF16):
    """MXFP4 skinny-M GEMM through a4w4_flatmm: a [M, K/2] packed E2M1 with M <= 128, b_shuffled from
    preshuffle_b_device on the packed weight bytes [N, K/2], both scale arrays in the MX_TILED layout."""
    r = None if n is None else _fast_gemm(_FLATMM4, a, b_shuffled, sfa_tiled, sfb_tiled, MX_TILED, c, c_dtype, n)
    if r is not None:
        return _done(r, "a4w4_flatmm")
    _need_torch()
    _check_operands(a, b_shuffled, 1, (2,), n=n)
    m, k = a.shape[-2], a.shape[-1] * 2
    if m <= 128:      # (more rows are the library's to refuse)
        _check_fp4_scales(sfa_tiled, sfb_tiled, MX_TILED, m, n, k)
    c, c_dtype = _out(c, (m, n), c_dtype, a.device)
    _check_ints("a4w4_flatmm", m, n, k, 2 * a.stride(-2), c.stride(-2))
    g = raw_gemm_args(a.data_ptr(), b_shuffled.data_ptr(), c.data_ptr(), sfa_tiled.data_ptr(), sfb_tiled.data_ptr(), m, n, k,
                      MX_TILED, c_dtype, stride_a=a.stride(-2) * 2, stride_b=k, stride_c=c.stride(-2), b_preshuffled=1)
    _check(lib().a4w4_flatmm(ctypes.byref(g), _stream()), "a4w4_flatmm")
    return c


def gemm_blockscale(a, b, sfa, sfb, c=None, c_dtype=FP32):
    """The reference's block-scale GEMM (1x128 / 128x128 scales), fp32 C by default as there."""
    r = _fast_gemm(_BLOCKSCALE, a, b, sfa, sfb, BLOCK, c, c_dtype, None)
    if r is not None:
        return _done(r, "a8w8_gemm_blockscale")
    g, c = _args_from_tensors(a, b, sfa, sfb, BLOCK, c, c_dtype, 0)
    _check(lib().a8w8_gemm_blockscale(ctypes.byref(g), _stream()), "a8w8_gemm_blockscale")
    return c


def flatmm(a, b_shuffled, sfa, sfb, n, scale_mode=ROWCOL, c=None, c_dtype=BF16):
    """Skinny-M GEMM over weights in the a8w8_preshuffle_b layout (flat u8 tensor of n*k bytes); scale_mode ROWCOL,
    TENSOR or MX_TILED (MXFP8: both scale arrays in the tiled layout)."""
    r = None if n is None else _fast_gemm(_FLATMM, a, b_shuffled, sfa, sfb, scale_mode, c, c_dtype, n)
    if r is not None:
        return _done(r, "a8w8_flatmm")
    g, c = _args_from_tensors(a, b_shuffled, sfa, sfb, scale_mode, c, c_dtype, 1, n=n)
    _check(lib().a8w8_flatmm(ctypes.byref(g), _stream()), "a8w8_flatmm")
    return c


def preshuffle_b(b_np):
    """Host pre-shuffle of a numpy [N, K] uint8 weight; returns a flat uint8 array."""
    import numpy as np
    b_np = np.ascontiguousarray(b_np, dtype=np.uint8)
    n, k = b_np.shape
    out = np.empty(n * k, np.uint8)
    _check(lib().a8w8_preshuffle_b(b_np.ctypes.data, out.ctypes.data, n, k), "a8w8_preshuffle_b")
    return out


def unshuffle_b(bs_np, n, k):
    import numpy as np
    bs_np = np.ascontiguousarray(bs_np, dtype=np.uint8)
    out = np.empty((n, k), np.uint8)
    _check(lib().a8w8_unshuffle_b(bs_np.ctypes.data, out.ctypes.data, n, k), "a8w8_unshuffle_b")
    return out


def preshuffle_b_device(b):
    _need_torch()
    n, k = b.shape
    _check_rows(b, "b", 1)
    if not b.is_contiguous():
        raise ValueError("b must be contiguous")
    out = torch.empty(n * k, dtype=torch.uint8, device=b.device)
    _check(lib().a8w8_preshuffle_b_device(b.data_ptr(), out.data_ptr(), n, k, _stream()), "a8w8_preshuffle_b_device")
    return out


def cvt_f32_to_e4m3(x, dialect=OCP, clamp240=False):
    r = _fast_encode(x, dialect, clamp240)
    if r is not None:
        return _done(r, "a8w8_cvt_f32_to_e4m3")
    _need_torch()
    x = x.contiguous()
    if x.dtype != torch.float32:
        raise TypeError(f"x must be float32, got {x.dtype}")
    if not x.is_cuda:
        raise ValueError("x must live on the GPU")
    out = torch.empty(x.shape, dtype=torch.uint8, device=x.device)
    _check(lib().a8w8_cvt_f32_to_e4m3(x.data_ptr(), out.data_ptr(), x.numel(), dialect, int(clamp240), _stream()),
           "a8w8_cvt_f32_to_e4m3")
    return out


def cvt_e4m3_to_f32(codes, dialect=OCP):
    r = _fast_decode(codes, dialect)
    if r is not None:
        return _done(r, "a8w8_cvt_e4m3_to_f32")
    _need_torch()
    codes = codes.contiguous()
    if codes.element_size() != 1:
        raise TypeError(f"codes must have elements of one byte, got {codes.dtype}")
    if not codes.is_cuda:
        raise ValueError("codes must live on the GPU")
    out = torch.empty(codes.shape, dtype=torch.float32, device=codes.device)
    _check(lib().a8w8_cvt_e4m3_to_f32(codes.data_ptr(), out.data_ptr(), codes.numel(), dialect, _stream()),
           "a8w8_cvt_e4m3_to_f32")
    return out


def quantize(x, scale_mode, group_rows=1):
    """fp32 [rows, K] -> (E4M3 bytes [rows, K], scales in the layout a8w8_gemm reads)."""
    r = _fast_quantize(x, scale_mode, group_rows)
    if r is not None:
        return _done(r, "a8w8_quantize")
    _need_torch()
    rows, k = x.shape
    _check_fp32_rows(x, "a8w8_quantize")
    q = torch.empty((rows, k), dtype=torch.uint8, device=x.device)
    if scale_mode == TENSOR:
        s = torch.empty(1, dtype=torch.float32, device=x.device)
    elif scale_mode == ROWCOL:
        s = torch.empty(rows, dtype=torch.float32, device=x.device)
    elif scale_mode == BLOCK and group_rows == 1:
        s = torch.empty((k // 128, rows), dtype=torch.float32, device=x.device)
    elif scale_mode == BLOCK:
        s = torch.empty((rows // 128, k // 128), dtype=torch.float32, device=x.device)
    elif scale_mode == MX:
        s = torch.empty((rows, k // 32), dtype=torch.uint8, device=x.device)
    elif scale_mode == MX_TILED:
        s = torch.empty(mx_tiled_bytes(rows, k), dtype=torch.uint8, device=x.device)
    else:
        raise A8W8Error(-6, "a8w8_quantize")
    _check(lib().a8w8_quantize(x.data_ptr(), rows, k, x.stride(0), q.data_ptr(), s.data_ptr(), scale_mode, group_rows,
                               _stream()), "a8w8_quantize")
    return q, s


def mx_tile_scales(sf, out=None):
    """Row-major E8M0 scales [rows, K/32] (u8, on the GPU) -> the MX_TILED layout (flat u8 tensor)."""
    _need_torch()
    rows, kb = sf.shape
    _check_rows(sf, "sf", 1)
    if out is not None and (not out.is_contiguous() or not out.is_cuda or out.numel() * out.element_size() < mx_tiled_bytes(rows, kb * 32)):
        raise ValueError(f"out must be a contiguous GPU tensor of {mx_tiled_bytes(rows, kb * 32)} bytes")
    if out is None:
        out = torch.empty(mx_tiled_bytes(rows, kb * 32), dtype=torch.uint8, device=sf.device)
    _check(lib().a8w8_mx_tile_scales(sf.data_ptr(), rows, kb * 32, sf.stride(0), out.data_ptr(), _stream()),
           "a8w8_mx_tile_scales")
    return out


def mx_tile_scales_ab(sfa, sfb):
    """Both scale arrays of a GEMM ([M, K/32] and [N, K/32] u8) -> MX_TILED, one launch."""
    _need_torch()
    m, kb = sfa.shape
    n = sfb.shape[0]
    _check_rows(sfa, "sfa", 1)
    _check_rows(sfb, "sfb", 1)
    if sfb.dim() != 2 or sfb.shape[1] < kb:
        raise ValueError(f"sfb must have rows of {kb} scales, got {tuple(sfb.shape)}")
    ta = torch.empty(mx_tiled_bytes(m, kb * 32), dtype=torch.uint8, device=sfa.device)
    tb = torch.empty(mx_tiled_bytes(n, kb * 32), dtype=torch.uint8, device=sfb.device)
    _check(lib().a8w8_mx_tile_scales_ab(sfa.data_ptr(), m, sfa.stride(0), ta.data_ptr(), sfb.data_ptr(), n,
                                        sfb.stride(0), tb.data_ptr(), kb * 32, _stream()), "a8w8_mx_tile_scales_ab")
    return ta, tb


def save_weights(path, b_np, scale_np, n, k, scale_mode, b_preshuffled=False):
    """Write quantised weights (numpy uint8, row-major [n, k] or pre-shuffled flat) and their scales to a file."""
    import numpy as np
    b_np = np.ascontiguousarray(b_np, dtype=np.uint8)
    scale_np = np.ascontiguousarray(scale_np)
    assert b_np.size == n * k and scale_np.nbytes == lib().a8w8_weight_scale_bytes(n, k, scale_mode)
    _check(lib().a8w8_weights_save(os.fsencode(path), b_np.ctypes.data, scale_np.ctypes.data, n, k, int(b_preshuffled),
                                   scale_mode), "a8w8_weights_save")


def load_weights(path):
    """-> (header, weights uint8 array, scales array: float32, or uint8 for the MX modes)."""
    import numpy as np
    h = WeightHeader()
    _check(lib().a8w8_weights_info(os.fsencode(path), ctypes.byref(h)), "a8w8_weights_info")
    b = np.empty(h.b_bytes, np.uint8)
    raw = np.empty(h.scale_bytes, np.uint8)
    _check(lib().a8w8_weights_load(os.fsencode(path), b.ctypes.data, b.nbytes, raw.ctypes.data, raw.nbytes), "a8w8_weights_load")
    scales = raw if h.scale_mode in (MX, MX_TILED) else raw.view(np.float32)
    return h, (b if h.b_preshuffled else b.reshape(h.n, h.k)), scales


def init(device=-1):
    """Explicit one-time set-up of a device (the current one by default); see a8w8_init."""
    _check(lib().a8w8_init(int(device)), "a8w8_init")


def kernel_name(g):
    r = lib().a8w8_kernel_name(ctypes.byref(g))
    return r.decode() if r else None
