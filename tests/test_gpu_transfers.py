"""Downloads on both sides of the line between the runtime's copy and the
chunked one (4 MiB), at chunk edges (1 MiB), and from several threads at once:
every value arrives."""
import threading

import numpy as np
import pytest

from cabanapd_amd import configs, engine
from cabanapd_amd._abi import make_desc
from tests.parity import ctx, say

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def cloud(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.random((n, 3))
    desc = make_desc("PMB", horizon=1e-4, K=1.0, dt=1e-7)
    w = configs._base(desc, x, np.full(n, 1e-9), 1.0, "cloud", 1e-4, 1)
    w["u"], w["v"] = rng.random((n, 3)), rng.random((n, 3))
    w["rho"] = rng.random(n) + 0.5
    s = engine.Spec(ctx(), desc, n)
    configs.upload(s, w)
    return s, w


@pytest.mark.parametrize("n", [4 * MIB // 24 - 1, 4 * MIB // 24 + 1, 5 * MIB // 24 + 1, 524287, 524288, 524289, 786433])
def test_downloads_at_chunk_edges(n):
    say(f"case: {n} particles, fields of {24 * n} and {8 * n} bytes")
    s, w = cloud(n, n)
    for fld in ("x", "u", "v", "rho"):
        assert np.array_equal(s.get(fld), w[fld]), fld
    s.close()


def test_downloads_from_several_threads():
    say("case: four specimens downloaded by four threads, ten times each")
    specs = [cloud(200000 + 31 * k, k) for k in range(4)]
    bad = []

    def read(s, w):
        for _ in range(10):
            for fld in ("u", "v"):
                if not np.array_equal(s.get(fld), w[fld]):
                    bad.append(fld)

    th = [threading.Thread(target=read, args=p) for p in specs]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    for s, _ in specs:
        s.close()
