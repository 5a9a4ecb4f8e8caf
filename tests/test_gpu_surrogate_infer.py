"""GPU tests of the inference kernel's queues: an answer is a function of its
query alone, so neither the number nor the order of the other queries, nor a
query with infinite or NaN inputs among them, may change a bit of it."""
import numpy as np
import pytest

from openshadinglanguage_amd import check, lib
from openshadinglanguage_amd import surrogate as S
from openshadinglanguage_amd import workloads as W

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sur():
    check(lib().oslmi_init())
    s = S.Surrogate(max_batch=2048)
    s.set_output_normalization([-0.5, -0.6, -0.7, -1.0], [1.3, 1.2, 1.1, 1.5])
    s.set_params(S.init_params(11))
    cells = np.zeros(S.NCELL, np.uint8)
    cells[7] = cells[20] = 1
    s.set_routing(cells)
    s.set_spot_check(0.2)  # a good part of an unfitted network's answers
    return s


def _infer(s, q, exact):
    n = q.shape[1]
    out = torch.full((4, n), -3.0, device="cuda:0")
    fbi = torch.empty(max(n, 1), dtype=torch.int32, device="cuda:0")
    fbn = torch.zeros(1, dtype=torch.int32, device="cuda:0")
    if exact:
        s.infer(q, out, material=W.layered_material(), fb_index=fbi, fb_count=fbn)
    else:
        s.infer(q, out)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("kind", ["upper", "sphere"])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 64, 65, 96, 127, 129, 4099, 300007])
def test_answers_do_not_depend_on_order(sur, n, kind, exact):
    make = S.upper_hemisphere_queries if kind == "upper" else W.surrogate_queries
    q = torch.from_numpy(make(n, 40)).to("cuda:0")
    print("infer %d %s exact=%s" % (n, kind, exact), flush=True)
    ref = _infer(sur, q, exact)
    assert not torch.any(ref == -3.0)
    perm = torch.randperm(n, device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(n))
    assert torch.equal(_infer(sur, q[:, perm].contiguous(), exact), ref[:, perm])
    k = (n + 1) // 2
    assert torch.equal(_infer(sur, q[:, :k].contiguous(), exact), ref[:, :k])


def test_bad_inputs_stay_in_their_query(sur):
    n = 1000
    q = torch.from_numpy(S.upper_hemisphere_queries(n, 41)).to("cuda:0")
    ref = _infer(sur, q, False)
    bad = torch.arange(3, n, 37, device="cuda:0")
    for row, v in ((0, float("nan")), (1, float("inf")), (3, float("-inf")), (2, float("nan"))):
        p = q.clone()
        p[row, bad] = v
        got = _infer(sur, p, False)
        good = torch.ones(n, dtype=torch.bool, device="cuda:0")
        good[bad] = False
        assert torch.equal(got[:, good], ref[:, good])
