"""The package's native call module (csrc/pycall.cpp) without a GPU: arguments
reach the C ABI in order (its own checks answer), and malformed calls raise."""
import numpy as np
import pytest

P = 4096            # a pointer that validation never follows
ST = (4, 4, 4, 1)


def test_prefill_calls_reach_the_abi_checks(nne):
    bad = (P, (2, 4, 16, 32), ST, P, (2, 2, 16, 32), ST, P, (2, 2, 16, 32), ST, P, ST, True)
    assert nne._native().flash(*bad, False, 0.0, 64, 64, None, 0) == nne.NNE_ESHAPE
    assert b"expected shape [2, 4, 16, 32], got [2, 2, 16, 32]" in nne.lib().nne_last_error()
    odd = bad[:1] + ((2, 3, 16, 32),) + bad[2:]
    assert nne._native().attention(*odd, 0, False, 0.0, None, 0) == nne.NNE_ESHAPE


def test_decode_calls_read_the_host_lengths(nne):
    lens = np.array([2, 5], np.int32)
    geo = (2, 1, 1, 5, 4, False, 0.0)
    rc = nne._native().decode_step(P, ST, P, P, P, lens, P, ST, P, ST, P, ST, *geo, None, 0)
    assert rc == nne.NNE_ECAPACITY and list(lens) == [2, 5]
    assert b"sequence 1 of length 5" in nne.lib().nne_last_error()
    rc = nne._native().decode_attention(P, ST, P, P, P, np.array([2, 6], np.int32), P, ST, *geo,
                                        None, 0)
    assert rc != nne.NNE_OK


def test_workspace_fields_are_checked(nne):
    lens = np.array([2], np.int32)
    rc = nne._native().decode_attention(P, ST, P, P, P, lens, P, ST, 1, 1, 1, 5, 4, False, 0.0,
                                        (P + 4, 1 << 20, P, 64), 0)
    assert rc == nne.NNE_EINVAL
    assert b"16-byte aligned" in nne.lib().nne_last_error()


@pytest.mark.parametrize("args", [(), ("x",), (P, (1, 2, 3)), (P, [1, 2, 3, 4]), (P, ST) * 20])
def test_malformed_calls_raise(nne, args):
    for fn in vars(nne._native()).values():
        with pytest.raises((TypeError, ValueError)):
            fn(*args)
