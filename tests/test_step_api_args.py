"""Arguments of the step-API coder that need no GPU: the exponential table in
every form it is taken in."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("form", ["list of int", "list of float", "int64", "uint64", "float64", "int64 tensor",
                                  "float64 tensor", "strided tensor"])
def test_lut_forms_keep_every_value(form):
    """Table entries go to 2**38; float32, which torch makes of a list of
    floats, holds 24 bits of them."""
    from sigcomp_amd.gpu_entropy_coding import _lut_on
    lut = np.array([(1 << 38) - 1 - 1234567 * k for k in range(256)], np.int64)
    arg = {"list of int": lut.tolist(), "list of float": [float(x) for x in lut], "int64": lut,
           "uint64": lut.astype(np.uint64), "float64": lut.astype(np.float64), "int64 tensor": torch.from_numpy(lut),
           "float64 tensor": torch.from_numpy(lut.astype(np.float64)),
           "strided tensor": torch.from_numpy(np.stack([lut, lut], 1))[:, 0]}[form]
    got = _lut_on(arg, torch.device("cpu"))
    assert got.dtype == torch.int64 and got.is_contiguous() and np.array_equal(got.numpy(), lut)


def test_lut_of_another_shape_is_refused():
    from sigcomp_amd.gpu_entropy_coding import _lut_on
    with pytest.raises(ValueError, match="256"):
        _lut_on([1] * 255, torch.device("cpu"))
