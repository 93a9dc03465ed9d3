"""The gradient list and its plans under host ASan + UBSan + LeakSanitizer
(tests/host_sanitize/gradient_list.cpp): the host stage on the CPU, the entry
points end to end on the GPU."""
import pytest

from test_host_sanitize import _run


def test_gradient_list_host_stage():
    _run("gradient_host", "gradient_list ok")


@pytest.mark.gpu
def test_gradient_list_end_to_end():
    _run("gradient_sanitize", "gradient_list ok")
