"""Device-tensor front end of the C ABI: torch supplies device memory and streams,
every computation happens in the HIP kernels of libaccera_mi355x.so."""
import ctypes
import struct

import torch

from . import _lib, tuned

_TORCH_TYPES = {
    torch.float32: _lib.F32, torch.float16: _lib.F16, torch.bfloat16: _lib.BF16,
    torch.int8: _lib.I8, torch.int32: _lib.I32, torch.int16: _lib.I16,
}


def _mat(t, name):
    strides = t.stride()
    if len(strides) not in (2, 3):
        raise ValueError(f"{name} must be 2-D, or 3-D for a batch")
    if not t.is_cuda:
        raise ValueError(f"{name} must live on the GPU (there is no CPU path)")
    return (t.data_ptr(), *strides) if len(strides) == 3 else (t.data_ptr(), 0, *strides)


def _problem(A, B, C):
    """(in type, out type, batch, M, N, K, A ptr + strides, B ..., C ...) of a 2-D call or of a batch
    (3-D tensors (batch, rows, cols); a 2-D A or B is shared by every problem of the batch)."""
    a_shape, b_shape, c_shape = A.shape, B.shape, C.shape
    batch = 1
    if len(a_shape) != 2 or len(b_shape) != 2 or len(c_shape) != 2:
        batch = c_shape[0] if len(c_shape) == 3 else 1
        if len(c_shape) == 2 and (len(a_shape) == 3 or len(b_shape) == 3):
            raise ValueError("a batched A or B needs a 3-D C")
        for t, name in ((A, "A"), (B, "B")):
            if t.dim() == 3 and t.shape[0] != batch:
                raise ValueError(f"{name} has {t.shape[0]} matrices, C has {batch}")
        a_shape, b_shape, c_shape = a_shape[-2:], b_shape[-2:], c_shape[-2:]
    M, K = a_shape
    K2, N = b_shape
    if K2 != K or c_shape != (M, N):
        raise ValueError(f"shape mismatch: A {tuple(A.shape)}, B {tuple(B.shape)}, C {tuple(C.shape)}")
    dtype = A.dtype
    in_type, out_type = _TORCH_TYPES.get(dtype), _TORCH_TYPES.get(C.dtype)
    if B.dtype != dtype or in_type is None or out_type is None:
        raise ValueError(f"unsupported dtypes {A.dtype}, {B.dtype}, {C.dtype}")
    return (in_type, out_type, batch, M, N, K, *_mat(A, "A"), *_mat(B, "B"), *_mat(C, "C"))


# (a raw handle without a stream object around it, a microsecond less per call; torch does not document it, so it may be missing)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _current_stream(C):
    """Raw hipStream_t of the stream that is current on C's device."""
    return _raw_stream(C.get_device()) if _raw_stream else torch.cuda.current_stream(C.device).cuda_stream


_pack = struct.Struct("19qdqd3q").pack  # acc950_gemm_call


class GemmCall:
    """One matmul+epilogue bound to its tensors, like one function of a package bound to
    its arrays: everything about the call is fixed at construction, calling it only
    launches.  Keeps the tensors alive; `stream` is a raw hipStream_t (int) or None for the
    stream that is current when the object is built."""

    def __init__(self, A, B, C, prologue=_lib.PROLOGUE_SET0, epilogue=_lib.EPILOGUE_RELU, variant=_lib.VARIANT_AUTO,
                 k_splits=0, stream=None, prologue_arg=0.0, epilogue_arg=0.0):
        problem = _problem(A, B, C)
        hit = None
        if variant == _lib.VARIANT_AUTO and k_splits == 0 and problem[2] == 1:
            # a recorded choice for this very shape (accera_amd.tune --save) goes before the library's cost model
            hit = tuned.lookup(problem[0], problem[1], problem[3], problem[4], problem[5], problem[8:10], problem[12:14], problem[16:18],
                               tuned.ops_class(prologue, prologue_arg, epilogue))
            if hit:
                variant, k_splits = hit
        if stream is None:
            stream = _current_stream(C)
        self.variant, self.k_splits = variant, k_splits  # as asked of the library (after the table look-up)
        self.tensors = (A, B, C)
        L = _lib.lib()
        handle = ctypes.c_int(-1)
        rc = L.acc950_bind(*problem, prologue, float(prologue_arg), epilogue, float(epilogue_arg), variant, k_splits, stream,
                           ctypes.byref(handle))
        if rc and hit:
            # the recorded kernel does not take this call after all (pointer alignment, ops): the library chooses
            self.variant, self.k_splits = _lib.VARIANT_AUTO, 0
            rc = L.acc950_bind(*problem, prologue, float(prologue_arg), epilogue, float(epilogue_arg), _lib.VARIANT_AUTO, 0, stream,
                               ctypes.byref(handle))
        _lib.check(rc)
        self._handle = handle.value
        self._launch, self._unbind = L.acc950_launch, L.acc950_unbind
        # what the library bound for this very call (its ops and pointers): kernel variant and number of K slices
        v, ks = ctypes.c_int(), ctypes.c_int()
        _lib.check(L.acc950_bound_choice(self._handle, ctypes.byref(v), ctypes.byref(ks)))
        self.chosen = (v.value, ks.value)

    def __call__(self):
        rc = self._launch(self._handle)
        if rc:
            _lib.check(rc)
        return self.tensors[2]

    def __del__(self):
        if getattr(self, "_handle", -1) >= 0:
            self._unbind(self._handle)
            self._handle = -1


def gemm_relu(A, B, C, prologue=_lib.PROLOGUE_SET0, epilogue=_lib.EPILOGUE_RELU, variant=_lib.VARIANT_AUTO,
              k_splits=0, stream=None, prologue_arg=0.0, epilogue_arg=0.0):
    """C = epilogue(prologue(C) + A @ B), in place on C, asynchronously.

    prologue: NONE keeps C, SET replaces it by ``prologue_arg`` (0: the fused matmul+ReLU),
    SCALE multiplies it by ``prologue_arg`` (GEMM beta); epilogue: NONE, RELU, RELU_NOCOND,
    SCALE by ``epilogue_arg`` (GEMM alpha), SET
    (/root/reference/docs/Tutorials/GPU/Tensor_MatMul_ElementWiseOps_GPU.md:85-99).

    A (M,K), B (K,N), C (M,N) are CUDA/HIP tensors; strides are honoured (a
    column-major B is ``B_storage.t()`` of an (N,K) tensor).  With a 3-D C (batch, M, N) the
    call is a batch of independent problems in one launch (the reference's batch matmul nest,
    /root/reference/accera/python/accera/test/mfma_tests.py:435-549); A and B are 3-D, or 2-D to be
    shared by the whole batch.  Types: fp16/bf16 in -> fp32/fp16/bf16 out, int8 -> int32/int16/int8,
    fp32 -> fp32.  Mirrors calling one function of an Accera package on (A, B, C)
    (/root/reference/README.md:124-130), on device memory.
    """
    problem = _problem(A, B, C)
    hit = None
    if variant == _lib.VARIANT_AUTO and k_splits == 0 and problem[2] == 1:
        # a recorded choice, as for a GemmCall; if the library refuses it for this call, its own choice runs
        in_type, out_type, _, M, N, K, _, _, a_rs, a_cs, _, _, b_rs, b_cs, _, _, c_rs, c_cs = problem
        hit = tuned.recorded(in_type, out_type, M, N, K, a_rs, a_cs, b_rs, b_cs, c_rs, c_cs, tuned.ops_class(prologue, prologue_arg, epilogue))
        if hit:
            variant, k_splits = hit
    if stream is None:
        stream = _current_stream(C)
    elif isinstance(stream, ctypes.c_void_p):
        stream = stream.value or 0
    run = _lib.lib().acc950_gemm_packed
    rc = run(_pack(*problem, prologue, prologue_arg, epilogue, epilogue_arg, variant, k_splits, stream))
    if rc == _lib.UNSUPPORTED and hit:
        rc = run(_pack(*problem, prologue, prologue_arg, epilogue, epilogue_arg, _lib.VARIANT_AUTO, 0, stream))
    if rc:
        _lib.check(rc)
    return C
