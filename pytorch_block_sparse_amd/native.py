"""ctypes binding of libpbs_hip.so, the C-ABI HIP library behind the three block-sparse matmuls.

This takes the place of the reference's pybind11 module ``block_sparse_native``
(native/block_sparse_native.cpp:31-34): tensors are passed as raw device pointers plus
sizes, kernels are launched on torch's current stream, and a non-zero return code raises
(the reference drops the code, block_sparse.py:565, :640).

There is no fallback: if the library is missing or the tensors are not on a GPU the calls
raise.
"""
import ctypes
import os

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "csrc", "libpbs_hip.so")

ABI_VERSION = 10   # PBS_ABI_VERSION of the header that the prototypes below restate

DTYPE_CODES = {torch.float32: 0, torch.bfloat16: 1}
SUPPORTED_DTYPES = tuple(DTYPE_CODES)

_lib = None

_vp = ctypes.c_void_p
_i32 = ctypes.c_int
_i64 = ctypes.c_int64

_PROTOTYPES = {
    "pbs_abi_version": (ctypes.c_int, []),
    "pbs_error_string": (ctypes.c_char_p, [_i32]),
    "pbs_build_indices": (_i32, [_vp, _vp, _i32, _i32, _i32, _vp, _vp, _vp, _vp, _vp, _vp, _vp]),
    "pbs_replace_blocks_workspace_bytes": (ctypes.c_size_t, [_i32, _i32, _i32]),
    "pbs_replace_blocks": (_i32, [_vp, _vp, _i32, _i32, _i32, _i32, _vp, _vp, _vp, _vp, _vp, _vp, _vp, ctypes.c_size_t, _vp]),
    "pbs_validate_indices_workspace_bytes": (ctypes.c_size_t, [_i32]),
    "pbs_validate_indices": (_i32, [_vp, _vp, _vp, _vp, _vp, _i32, _i32, _i32, _vp, _vp, ctypes.c_size_t, _vp]),
    "pbs_blocksparse_matmul_plan_bytes": (ctypes.c_size_t, [_i32, _i32]),
    "pbs_blocksparse_matmul_plan": (_i32, [_vp, _vp, _i32, _i32, _i32, _vp, ctypes.c_size_t, _vp]),
    "pbs_blocksparse_matmul_plan_part_bytes": (ctypes.c_size_t, [_i32, _i32]),
    "pbs_blocksparse_matmul_plan_part": (_i32, [_vp, _vp, _i32, _i32, _i32, _i32, _vp, ctypes.c_size_t, _vp]),
    "pbs_blocksparse_derive": (
        _i32,
        [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _vp, ctypes.c_size_t, _vp, ctypes.c_size_t, _vp, ctypes.c_size_t, _vp],
    ),
    "pbs_blocksparse_matmul_part": (_i32, [_i64, _i32, _i32, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul": (_i32, [_vp, _vp, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _i32, _i32, _vp]),
    "pbs_blocksparse_matmul_workspace_bytes": (ctypes.c_size_t, [_i64, _i32, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul_parts_bytes": (ctypes.c_size_t, [_i64, _i32, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul_ws": (
        _i32,
        [_vp, _vp, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _i32, _i32, _vp, ctypes.c_size_t, _vp],
    ),
    "pbs_blocksparse_matmul_back_workspace_bytes": (ctypes.c_size_t, [_i64, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul_back": (
        _i32,
        [_vp, _vp, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _i32, _vp, ctypes.c_size_t, _vp],
    ),
    "pbs_blocksparse_matmul_back_units_bytes": (ctypes.c_size_t, [_i64, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul_back_units": (_i32, [_vp, _vp, _i32, _i32, _i32, _vp, ctypes.c_size_t, _vp]),
    "pbs_blocksparse_matmul_back_bias_workspace_bytes": (ctypes.c_size_t, [_i64, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul_back_bias": (
        _i32,
        [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _i32, _vp, ctypes.c_size_t, _vp],
    ),
    "pbs_blocksparse_linear_back_workspace_bytes": (ctypes.c_size_t, [_i64, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_linear_back": (
        _i32,
        [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _i32, _vp, ctypes.c_size_t, _vp],
    ),
    "pbs_blocksparse_matmul_back_blocks_workspace_bytes": (ctypes.c_size_t, [_i64, _i32, _i32, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul_back_blocks": (
        _i32,
        [_vp, _i32, _vp, _i32, _vp, _i64, _i32, _i32, _vp, _i32, _i32, _vp, ctypes.c_size_t, _vp],
    ),
    "pbs_blocksparse_matmul_back_noalloc_max_bytes": (ctypes.c_size_t, []),
    "pbs_blocksparse_matmul_back_noalloc_init": (_i32, []),
    "pbs_protocol_failures": (_i32, [ctypes.POINTER(ctypes.c_uint)]),
    "pbs_blocksparse_matmul_kernel_name": (ctypes.c_char_p, [_i64, _i32, _i32, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul_kernel_form": (ctypes.c_char_p, [_i64, _i32, _i32, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul_back_kernel_name": (ctypes.c_char_p, [_i64, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul_back_kernel_form": (ctypes.c_char_p, [_i64, _i32, _i32, _i32, _i32]),
    "pbs_blocksparse_matmul_back_noalloc": (_i32, [_vp, _vp, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _i32, _vp]),
}

EXPORTED_SYMBOLS = tuple(_PROTOTYPES)


class NativeLibraryMissing(ImportError):
    pass


def load():
    """Load libpbs_hip.so (once) and declare the prototypes of its entry points."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise NativeLibraryMissing(
            f"{LIB_PATH} is not built. Run `python -m pytorch_block_sparse_amd.csrc.build` "
            f"(or `make -C {os.path.dirname(LIB_PATH)}`); there is no non-HIP path for the matmuls."
        )
    lib = ctypes.CDLL(LIB_PATH)
    for name, (restype, argtypes) in _PROTOTYPES.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    if lib.pbs_abi_version() != ABI_VERSION:
        raise NativeLibraryMissing(f"{LIB_PATH} is version {lib.pbs_abi_version()}, expected {ABI_VERSION}: build it again")
    _lib = lib
    return lib


_torch_path = None


def torch_path():
    """The extension module csrc/_pbs_torch.so: the products on torch tensors (result and workspace allocation, plans,
    autograd node) on top of the C ABI.  Loaded on first use; like the library it has no stand-in."""
    global _torch_path
    if _torch_path is None:
        load()
        try:
            from .csrc import _pbs_torch
        except ImportError as e:
            raise NativeLibraryMissing(
                f"{_HERE}/csrc/_pbs_torch.so cannot be loaded ({e}). Run `python -m pytorch_block_sparse_amd.csrc.build`."
            ) from e
        _torch_path = _pbs_torch
    return _torch_path


def error_string(code):
    return load().pbs_error_string(int(code)).decode()


def _check(code, what):
    if code != 0:
        raise RuntimeError(f"{what} failed with code {code}: {error_string(code)}")


def check_protocol(what):
    """With PBS_DEBUG set: raise if a bounded wait of a barrier-free kernel has run out on the current device since the last check
    (the kernel marks the affected results NaN and counts the event; without this the call reports success).  The products of
    ``torch_path()`` check by themselves."""
    if os.environ.get("PBS_DEBUG"):
        torch_path().check_protocol(what)


def matmul_kernel_name(tokens, n, k, nnz, transpose, dtype, with_workspace=True):
    """Which kernel pbs_blocksparse_matmul_ws runs for these sizes (for benchmark labels)."""
    return load().pbs_blocksparse_matmul_kernel_name(
        tokens, n, k, nnz, 1 if transpose else 0, DTYPE_CODES[dtype], 1 if with_workspace else 0).decode()


def matmul_kernel_form(tokens, n, k, nnz, transpose, dtype, with_workspace=True):
    """That name and in which of its forms the kernel runs (for tests of a form)."""
    return load().pbs_blocksparse_matmul_kernel_form(
        tokens, n, k, nnz, 1 if transpose else 0, DTYPE_CODES[dtype], 1 if with_workspace else 0).decode()


def matmul_back_kernel_name(tokens, out_features, in_features, nnz, dtype):
    return load().pbs_blocksparse_matmul_back_kernel_name(tokens, out_features, in_features, nnz, DTYPE_CODES[dtype]).decode()


def matmul_back_kernel_form(tokens, out_features, in_features, nnz, dtype):
    return load().pbs_blocksparse_matmul_back_kernel_form(tokens, out_features, in_features, nnz, DTYPE_CODES[dtype]).decode()


def _stream(index=None):
    """The current stream of device `index` (default: the current device) as a hipStream_t."""
    if index is None:
        index = torch.cuda.current_device()
    raw = getattr(torch._C, "_cuda_getCurrentRawStream", None)   # the handle without a Stream object around it
    return ctypes.c_void_p(raw(index) if raw is not None else torch.cuda.current_stream(index).cuda_stream)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None and t.numel() > 0 else ctypes.c_void_p(0)


def _require_cuda(*tensors):
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError(
                "pytorch_block_sparse_amd: the block-sparse matmuls run only on a GPU through libpbs_hip.so; "
                f"got a tensor on {t.device}"
            )


def build_indices(block_mask, block_ptr, nnz):
    """Device build of (blocks, cols_a, row_start_ends_a, rows_b, col_start_ends_b) for a CUDA mask."""
    lib = load()
    _require_cuda(block_mask, block_ptr)
    X, Y = block_mask.shape
    dev = block_mask.device
    mask_u8 = block_mask.contiguous().view(torch.uint8) if block_mask.dtype == torch.bool else (
        block_mask != 0
    ).contiguous().view(torch.uint8)
    if block_ptr is not None:
        block_ptr = block_ptr.to(device=dev, dtype=torch.int64).contiguous()
        if block_ptr.numel() != nnz:
            raise RuntimeError(f"block_ptr has {block_ptr.numel()} entries for {nnz} blocks")
    i32 = dict(dtype=torch.int32, device=dev)
    cols_a = torch.empty((nnz, 2), **i32)
    rows_b = torch.empty((nnz, 2), **i32)
    blocks = torch.empty((2 * nnz,), **i32)
    row_ptr = torch.empty((X + 1,), **i32)
    col_ptr = torch.empty((Y + 1,), **i32)
    status = torch.zeros((2,), **i32)
    with torch.cuda.device(dev):
        code = lib.pbs_build_indices(
            _ptr(mask_u8), _ptr(block_ptr), X, Y, nnz, _ptr(cols_a), _ptr(row_ptr), _ptr(rows_b), _ptr(col_ptr),
            _ptr(blocks), _ptr(status), _stream(),
        )
    _check(code, "pbs_build_indices")
    counted, err = status.tolist()
    if err == 1:
        raise RuntimeError(f"block mask holds {counted} blocks but {nnz} were expected")
    if err == 2:
        raise RuntimeError("block_ptr holds an entry outside [0, n_blocks)")
    return blocks, cols_a, row_ptr, rows_b, col_ptr


def blocksparse_matmul_plan(ptr, indices, n, k):
    """Schedule buffer of the dense x block-sparse product for (ptr, indices); depends on the pattern only."""
    lib = load()
    _require_cuda(ptr, indices)
    nbytes = lib.pbs_blocksparse_matmul_plan_bytes(n, k)
    plan = torch.empty((nbytes // 4,), dtype=torch.int32, device=ptr.device)
    with torch.cuda.device(ptr.device):
        code = lib.pbs_blocksparse_matmul_plan(
            _ptr(ptr), _ptr(indices), n, k, indices.shape[0], _ptr(plan), nbytes, _stream()
        )
    _check(code, "pbs_blocksparse_matmul_plan")
    return plan


def _dtype_code(t):
    code = DTYPE_CODES.get(t.dtype)
    if code is None:
        raise RuntimeError(f"unsupported dtype {t.dtype}; supported: {SUPPORTED_DTYPES}")
    return code


def blocksparse_matmul(dense_a, data, plan, n, k, nnz, transpose, bias=None, out=None):
    """out[tokens, n] = dense_a[tokens, k] . W^T (transpose) or . W (not transpose), with a plan of blocksparse_matmul_plan."""
    lib = load()
    _require_cuda(dense_a, data, plan, bias)
    code_dtype = _dtype_code(dense_a)
    if data.dtype != dense_a.dtype:
        raise RuntimeError(f"dense operand is {dense_a.dtype} but the block data is {data.dtype}")
    if bias is not None and bias.dtype != dense_a.dtype:
        raise RuntimeError(f"bias is {bias.dtype}, expected {dense_a.dtype}")
    tokens, tr = dense_a.shape[0], 1 if transpose else 0
    if out is None:
        out = torch.empty((tokens, n), dtype=dense_a.dtype, device=dense_a.device)
    # the transposed copy of the blocks that the forward bf16 kernel for dense patterns works from, or the bf16 parts of the blocks that
    # larger fp32 products are made of (both made by the library)
    ws_bytes = (lib.pbs_blocksparse_matmul_workspace_bytes(tokens, n, k, nnz, tr, code_dtype)
                or lib.pbs_blocksparse_matmul_parts_bytes(tokens, n, k, nnz, tr, code_dtype))
    ws = torch.empty((ws_bytes,), dtype=torch.uint8, device=dense_a.device)
    with torch.cuda.device(dense_a.device):
        code = lib.pbs_blocksparse_matmul_ws(
            _ptr(dense_a), _ptr(data), _ptr(plan), _ptr(bias), _ptr(out), tokens, n, k, nnz, tr, code_dtype, _ptr(ws), ws_bytes, _stream(),
        )
        _check(code, "pbs_blocksparse_matmul_ws")
        check_protocol("pbs_blocksparse_matmul_ws")
    return out


def blocksparse_matmul_back(dense_a, dense_b, row_start_ends_a, cols_a, out):
    """out (packed [nnz*32, 32]) = blocks of dense_a^T . dense_b on the pattern's support."""
    lib = load()
    _require_cuda(dense_a, dense_b, row_start_ends_a, cols_a, out)
    code_dtype = _dtype_code(dense_a)
    if dense_b.dtype != dense_a.dtype or out.dtype != dense_a.dtype:
        raise RuntimeError("operands and result must share one dtype")
    tokens, out_features = dense_a.shape
    sizes = (tokens, out_features, dense_b.shape[1], cols_a.shape[0], code_dtype)
    ws_bytes = lib.pbs_blocksparse_matmul_back_workspace_bytes(*sizes)
    ws = torch.empty((ws_bytes,), dtype=torch.uint8, device=dense_a.device)
    with torch.cuda.device(dense_a.device):
        code = lib.pbs_blocksparse_matmul_back(
            _ptr(dense_a), _ptr(dense_b), _ptr(row_start_ends_a), _ptr(cols_a), _ptr(out), *sizes, _ptr(ws), ws_bytes, _stream(),
        )
    _check(code, "pbs_blocksparse_matmul_back")
    return out
