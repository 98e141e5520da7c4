"""Calls that the library refuses on the host, before any device is needed."""

import pytest

import ludwig_amd as L


@pytest.fixture
def lib():
    lib = L.lib()
    lib.ldw_error_mode_set(0)
    yield lib
    lib.ldw_error_mode_set(1)


@pytest.mark.parametrize("c", [0, -1, -300])
def test_bias_gradient_without_channels(lib, c):
    # the launch divides by the channel count
    assert lib.ldw_nn_bias_grad(None, None, 10, c, 0) != 0
    assert f"{c} channels" in lib.ldw_last_error().decode()
