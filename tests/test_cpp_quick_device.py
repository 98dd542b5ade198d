"""The quick visibility test in the form that the device runs (tests/cpp/quick_device_test.cpp), on the CPU."""
from test_cpp_host import run


def test_device_form_decides_as_the_oracle():
    """Zeros, denormals, the limits of the bound, huge values, infinities and NaN in
    objects and views, with medians that drop a NaN operand as the device's do."""
    out = run("quick_device_test")
    assert "quick cull, device form: 0 failures" in out
