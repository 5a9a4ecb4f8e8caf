"""build() compiles kernels that only tests run ahead of time, but does not
depend on them: a tests directory without a program set, or with one of
another form, leaves those kernels to their first use (no GPU needed)."""
import os
import subprocess
import sys

import pytest

import __graft_entry__ as E


@pytest.mark.parametrize("tests", [(), ("_gsprogs.py", "_mxprogs.py", "_pnprogs.py")],
                         ids=["missing", "other form"])
def test_build_does_not_need_the_test_programs(tmp_path, tests):
    # a tree of the entry point, the package and another tests directory
    with open(E.__file__) as f:
        (tmp_path / "__graft_entry__.py").write_text(f.read())
    os.symlink(os.path.join(E.ROOT, "openshadinglanguage_amd"), tmp_path / "openshadinglanguage_amd")
    (tmp_path / "tests").mkdir()
    for name in tests:
        (tmp_path / "tests" / name).write_text("")
    jobs = ["tests:" + s for s in E.TEST_SETS]
    code = "import __graft_entry__ as E; E._compile(%r, optional=%r)" % (jobs, jobs)
    r = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    assert r.stdout.count("not compiled ahead") == len(jobs), r.stdout


def test_a_failed_job_of_the_framework_fails_the_build():
    with pytest.raises(RuntimeError, match="unknown job"):
        E._compile(["nothing"])
