"""The default shape of a propagation plan's tiles (tests/cpp/tree_shape_test.cpp), on the CPU."""
from test_cpp_host import run


def test_shallow_trees_take_few_steps():
    out = run("tree_shape_test")
    assert "trees, 0 failures" in out
