"""Error paths of the host driver, on a stand-in for the HIP runtime (no GPU):
calls that fail midway leave nothing behind that a later call would trip over."""
import pytest

from fake_hip import run

@pytest.mark.parametrize("call", ["g.enum(MOT, 100, 8_000_000)", "abi.time_order(np.zeros(8_000_000, np.int32))",
                                  "graph(200_000, 900)"])
def test_an_error_is_told_once(call):
    """Memory that ran out in one call is not the next call's error."""
    run("""
g = graph()
fake.fake_limit(fake.fake_used() + (64 << 20))
fails(lambda: %s, 4)
g.count(MOT, 100)
fake.fake_limit(1 << 40)
%s
g.close()
""" % (call, call))
