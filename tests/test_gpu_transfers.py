"""Downloads on both sides of the line between the runtime's copy and the
chunked one (4 MiB), at chunk edges (1 MiB), and from several threads at once:
every value arrives."""
import threading
import time

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


def test_download_does_not_wait_for_other_specimens():
    """A download of a specimen whose stream has much queued waits for that
    work alone: another specimen's download goes through meanwhile."""
    n_side = 80
    x, vol, _ = configs.grid_cell_centred([0, 0, 0], [1.0] * 3, (n_side,) * 3)
    desc = make_desc("PMB", horizon=3.01 / n_side, K=1.0, dt=1e-7, fracture=True, G0=1.0)
    w = configs._base(desc, x, vol, 1.0, "busy", 1.0 / n_side, 1)
    busy = engine.Spec(ctx(), desc, x.shape[0])
    configs.upload(busy, w)
    configs.setup(busy, w)
    # streams share a few hardware queues in turn: of four specimens some are
    # not on the busy one's
    idle = [cloud(200000, k) for k in range(4)]
    for s in [busy] + [s for s, _ in idle]:
        s.get("u")  # slots, workers and staging are there
    took = {}

    def read(name, s):
        t = time.perf_counter()
        s.get("u")
        took[name] = time.perf_counter() - t

    for _ in range(600):
        busy.compute_energy_async()
    th = [threading.Thread(target=read, args=a) for a in [("busy", busy)] + [(k, s) for k, (s, _) in enumerate(idle)]]
    th[0].start()
    time.sleep(0.005)
    for t in th[1:]:
        t.start()
    for t in th:
        t.join()
    best = min(took[k] for k in range(4))
    say(f"case: downloads of 12 and 5 MB: behind 600 energy passes {1e3 * took['busy']:.1f} ms, "
        f"of idle specimens meanwhile from {1e3 * best:.1f} ms")
    assert took["busy"] > 0.04
    assert best < 0.5 * took["busy"]
    for s, w in idle:
        assert np.array_equal(s.get("u"), w["u"])
        s.close()
    busy.close()
