"""The eager ops' CPython module (binding/native.cpp) where a call is refused: every refusal is a RuntimeError. The tensors
claim a GPU without having one (wrapper subclasses, no storage), so the checks run on a machine without a GPU."""

import pytest
import torch

BF, I8, F32 = torch.bfloat16, torch.int8, torch.float32


class Claim(torch.Tensor):
    """A tensor of the given shape and type on "cuda:0", without storage."""

    @staticmethod
    def __new__(cls, *shape, dt=BF):
        return torch.Tensor._make_wrapper_subclass(cls, shape, dtype=dt, device="cuda:0")

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        raise NotImplementedError(str(func))


C = Claim
# op -> its arguments after one activation tensor x of the given shape and type, and where x goes
CALLS = {
    "gemv": ((1, 64), BF, lambda x: (C(16, 64, dt=I8), C(16, dt=F32), x, C(1, 16), 0)),
    "gemv_w4": ((1, 128), BF, lambda x: (C(8, 64, dt=torch.uint8), C(8, 1, dt=F32), x, C(1, 8), 0)),
    "gemv_w4z": ((1, 128), BF, lambda x: (C(8, 16, dt=torch.int32), C(8, 1, dt=torch.float16),
                                          C(8, 1, dt=torch.int32), x, C(1, 8), 0)),
    "silu_mul": ((2, 128), BF, lambda x: (x, C(2, 64))),
    "gemm_i8": ((2, 64), I8, lambda x: (x, C(2, dt=F32), C(8, 64, dt=I8), C(8, dt=F32), None, C(2, 8), False)),
    "gemm_i8_q": ((2, 64), I8, lambda x: (x, C(1, 2, dt=F32), C(64, 64, dt=I8), C(64, dt=F32), None, C(2, 64, dt=I8),
                                          C(1, 2, dt=F32), False)),
    "gemm_w8": ((2, 64), BF, lambda x: (x, C(8, 64, dt=I8), C(8, dt=F32), None, C(2, 8), False)),
    "quant_rows": ((2, 64), BF, lambda x: (x, C(2, 64, dt=I8), C(2, dt=F32))),
    "add_layernorm_q": ((2, 64), BF, lambda x: (x, None, C(64), C(64), C(2, 64, dt=I8), C(2, dt=F32), 1e-5, None)),
    "add_rmsnorm_q": ((2, 64), BF, lambda x: (x, None, C(64), C(2, 64, dt=I8), C(2, dt=F32), 1e-5, None)),
    "silu_mul_q": ((2, 128), BF, lambda x: (x, C(2, 64, dt=I8), C(2, dt=F32), None)),
}


@pytest.mark.parametrize("op", sorted(CALLS))
def test_a_tensor_without_a_pointer_is_an_error(op):
    """Under vmap an argument has no data pointer to read. The read throws, which must happen with the interpreter lock
    held (it ended the process when the lock had been released), so before anything asks for the stream."""
    from lfm2opt import _capi

    shape, dt, args = CALLS[op]

    def call(x):
        getattr(_capi.native(), op)(*args(x))
        return x

    with pytest.raises(RuntimeError, match="data pointer"):
        torch.func.vmap(call)(Claim(3, *shape, dt=dt))


@pytest.mark.parametrize("op", ["gemv_w4", "gemv_w4z"])
def test_w4_weights_without_columns_are_an_error(op):
    """K = 0 makes a group of no weights: refused before anything is divided by it."""
    from lfm2opt import _capi

    x, y = C(1, 0), C(1, 8)
    args = {"gemv_w4": (C(8, 0, dt=torch.uint8), C(8, 1, dt=F32), x, y, 0),
            "gemv_w4z": (C(8, 0, dt=torch.int32), C(8, 1, dt=torch.float16), C(8, 1, dt=torch.int32), x, y, 0)}[op]
    with pytest.raises(RuntimeError, match="group size must be a multiple of 32"):
        getattr(_capi.native(), op)(*args)


@pytest.mark.parametrize("op", ["gemv_w4_rmsnorm", "gemv_conv_rmsnorm"])
def test_w4z_weights_without_columns_are_an_error_with_a_norm(op):
    from lfm2opt.kernels import ext

    W, S, Z = C(24, 0, dt=torch.int32), C(24, 1, dt=torch.float16), C(24, 1, dt=torch.int32)
    args = {"gemv_w4_rmsnorm": (W, S, Z, C(1, 0), C(0), 1e-5, C(1, 24)),
            "gemv_conv_rmsnorm": (W, S, Z, C(1, 0), C(0), 1e-5, C(3, 1, 8), C(3, 8), None, C(2, dt=torch.int64), C(1, 8))}[op]
    with pytest.raises(RuntimeError, match="group size must be a multiple of 32"):
        getattr(ext(), op)(*args)


@pytest.mark.parametrize("op", ["gemv_w4", "gemv_w4z"])
def test_w4_epilogue_as_a_float(op):
    """epi = 1.0 is 1 (the call goes on to read the pointers); another number is refused as an epilogue."""
    from lfm2opt import _capi

    shape, dt, args = CALLS[op]

    def call(x, epi):
        a = args(x)
        getattr(_capi.native(), op)(*a[:-2], C(1, 4), epi)
        return x

    with pytest.raises(RuntimeError, match="data pointer"):
        torch.func.vmap(lambda x: call(x, 1.0))(Claim(3, *shape, dt=dt))
    with pytest.raises(RuntimeError, match="epi 0"):
        call(C(*shape), 1.5)
