"""A graph with one broken rule is refused as a bad argument, with the rule's
name: by the check kernels where a GPU is visible, by the host's restatement of
them elsewhere."""
import numpy as np
import pytest

from oracle import prep
from helpers import random_graph

BROKEN = ["endpoint low", "endpoint high", "time", "out span", "in span", "out monotone", "in monotone", "out range",
          "in range", "out vertex", "in vertex", "out order", "in order"]
RULE = {"endpoint": "edge endpoint out of [0, V)", "time": "edges are not sorted by time",
        "span": "CSR offsets must span [0, E]", "monotone": "CSR offsets not monotone",
        "range": "CSR position out of range", "vertex": "CSR position on the wrong vertex",
        "order": "CSR positions not ascending"}


def broken(what, E):
    """A valid graph's arrays with the rule `what` violated somewhere in the middle."""
    rng = np.random.default_rng(E)
    U, V, T = random_graph(rng, E, max(4, E // 8), 4 * E)
    g = {k: np.array(v) if isinstance(v, np.ndarray) else v for k, v in prep.preprocess(U, V, T).items()}
    side = "in" if what.startswith("in ") else "out"
    P, R = g[side + "V"], g[side + "R"]
    eg = g["Eg"].reshape(-1, 3)
    deg = np.diff(R)
    x = int(np.argmax(deg))  # a list of several slots
    if what == "endpoint low":
        eg[E // 2, 0] = -1
    elif what == "endpoint high":
        eg[E // 2, 1] = g["V"]
    elif what == "time":
        eg[E // 2, 2] = eg[E - 1, 2] + 1
    elif what.endswith("span"):
        R[-1] -= 1
    elif what.endswith("monotone"):
        R[x + 1] = R[x] - 1 if R[x] > 0 else R[x + 2] + 1
    elif what.endswith("range"):
        P[E // 2] = E if E % 2 else -1
    elif what.endswith("vertex"):
        y = int(np.nonzero(deg)[0][0])
        y = y if y != x else int(np.nonzero(deg)[0][1])
        P[R[x]], P[R[y]] = P[R[y]], P[R[x]]
    elif what.endswith("order"):
        P[R[x]], P[R[x] + 1] = P[R[x] + 1], P[R[x]]
    return g


def check(what, E):
    from everest_amd import abi
    with pytest.raises(abi.TMError) as e:
        abi.DeviceGraph.from_dict(broken(what, E))
    print(what, E, e.value, flush=True)
    assert e.value.status == 1
    return str(e.value)


@pytest.mark.parametrize("what", BROKEN)
def test_refused_without_gpu(what):
    from everest_amd import abi
    if abi.lib().tm_device_count() > 0:
        pytest.skip("the check kernels run here")
    msg = check(what, 300)
    if "monotone" not in what:  # (offsets that step back break the lists around them too)
        assert RULE[what.split()[-1] if what.split()[0] in ("in", "out") else what.split()[0]] in msg


@pytest.mark.gpu
@pytest.mark.parametrize("E", [40, 257, 5000])
@pytest.mark.parametrize("what", BROKEN)
def test_refused_on_gpu(what, E):
    msg = check(what, E)
    assert RULE[what.split()[-1] if what.split()[0] in ("in", "out") else what.split()[0]] in msg
