"""The committed include/rocrand/rocrand_amd_mathtab.h is what its generator writes."""
import importlib.util
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TAB = os.path.join(ROOT, "include", "rocrand", "rocrand_amd_mathtab.h")
MAKE = os.path.join(ROOT, "rocrand_amd", "data", "make_math_tables.py")


def test_tables_match_generator(tmp_path):
    """The committed header is what make_math_tables.py writes."""
    spec = importlib.util.spec_from_file_location("make_math_tables", MAKE)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    mod.OUT = str(tmp_path / "rocrand_amd_mathtab.h")
    mod.main()
    with open(TAB) as a, open(mod.OUT) as b:
        assert a.read() == b.read()
