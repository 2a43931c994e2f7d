"""Which kernels a dynamically quantized layer may take: the host's decisions, without a GPU."""

import numpy as np
import pytest

import lucid_amd as L
import lucid_amd.nn.quantized.dynamic as nnqd
from lucid_amd.nn.module import Module
from lucid_amd.nn.quantized.dynamic import linear as dl


def _layer(N, K, **other):
    """A layer whose buffers are host tensors."""
    lin = object.__new__(nnqd.Linear)
    Module.__init__(lin)
    lin.in_features, lin.out_features = K, N
    bufs = dict(weight_int8=np.zeros((N, K), np.int8), weight_scale=np.ones(N, np.float32),
                weight_zero_point=np.zeros(N, np.float32), bias=np.zeros(N, np.float32))
    for name, v in {**bufs, **other}.items():
        lin.register_buffer(name, v if v is None or isinstance(v, L.Tensor) else L.Tensor.from_numpy(v, "cpu"))
    return lin


@pytest.mark.parametrize("other,takes", [
    ({}, True), ({"bias": None}, True),
    ({"weight_int8": np.zeros((8, 31), np.int8)}, False), ({"weight_int8": np.zeros((7, 32), np.int8)}, False),
    ({"weight_int8": np.zeros(8 * 32, np.int8)}, False), ({"weight_int8": np.zeros((8, 32), np.int16)}, False),
    ({"weight_scale": np.ones(7, np.float32)}, False), ({"weight_scale": np.ones(8, np.float16)}, False),
    ({"bias": np.zeros(7, np.float32)}, False), ({"bias": np.zeros(8, np.float16)}, False),
    ({"bias": np.zeros(8, np.float64)}, False),
    ({"weight_int8": L.Tensor((8, 32), L.int8, "cpu", host=np.zeros((8, 32), np.int8), offset=4)}, False),
])
def test_kernels_read_by_address_only_what_they_expect(other, takes):
    """Sizes, types and the weight's alignment: all else is left to the operators that check."""
    assert (dl._kernel_operands(_layer(8, 32, **other), 8, 32) is not None) is takes


@pytest.mark.parametrize("M,K,takes", [
    (1, 1, True), (1, 131071, False), (1, 131007, True), (1, 131056, True), (1, 131072, False),
    # 64-byte rows of a short K: far fewer of them than M * K suggests
    (1 << 22, 3, True), ((1 << 22) + 1, 3, False), (1 << 26, 3, False), (1 << 26, 17, False), (1 << 22, 64, True),
    ((1 << 22) + 1, 64, False), ((1 << 21), 127, True), ((1 << 21) + 1, 127, False), (1 << 24, 16, True), (1 << 27, 16, False),
])
def test_one_call_is_for_codes_that_fit_its_rows_and_scratch(M, K, takes):
    assert dl._one_call_takes(M, K) is takes
    if takes:  # what the call itself refuses: padded codes in whole blocks of 8192 from 2^32 on, rows beyond 131071
        ld = dl._code_row_bytes(K)
        assert ld % 16 == 0 and K <= ld <= 131071 and (M * ld + 8191) // 8192 * 8192 < 1 << 32


def test_a_copied_type_is_the_type():
    import copy
    from lucid_amd import _tensor as T
    for dt in T._ALL:
        assert copy.deepcopy([dt])[0] is dt and copy.copy(dt) is dt


def test_another_weight_forgets_what_was_derived_from_the_last():
    """Assigned, registered or loaded: the row sums and padded rows are those of the weight that is there."""
    lin = _layer(8, 30)
    new = L.Tensor.from_numpy(np.ones((8, 30), np.int8), "cpu")
    for replace in (lambda: setattr(lin, "weight_int8", new), lambda: lin.register_buffer("weight_int8", new),
                    lambda: lin.load_state_dict({"weight_int8": new}, strict=False)):
        lin._wsum = lin._wrows = "of the last weight"
        replace()
        assert lin._wsum is None and lin._wrows is None
    lin._wsum = "of this weight"
    lin.bias = None
    assert lin._wsum == "of this weight"
