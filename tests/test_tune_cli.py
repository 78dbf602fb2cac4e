"""A tuning table is read only by programs that load it: the tuner writes none into the package, and the bench loads none."""
import os

from birp_cpp_amd import tune

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_tuner_writes_outside_the_package():
    out = tune.parser().parse_args([]).out
    assert os.path.dirname(os.path.abspath(out)) != os.path.join(ROOT, "birp_cpp_amd")
    assert not os.path.isabs(out)


def test_the_bench_measures_the_library_s_own_choice():
    with open(os.path.join(ROOT, "bench.py")) as f:
        assert "autotune_load" not in f.read()
