"""Results around the sizes where their last 2 MiB are cut in halves (csrc/readback.hip), on the host alone: every byte arrives, in
one piece and in several, the second and later results over earlier ones in the same buffers."""
import pytest

from test_readback_host import Engine, host  # noqa: F401 - a fixture

K = 1024


@pytest.mark.parametrize("sizes", [(512 * K,), (512 * K + 16,), (1024 * K - 16,), (1024 * K,), (1024 * K + 16,), (1152 * K + 16, 32),
                                   (2048 * K - 16, 1024, 2048 * K + 48), (4096 * K,), (4096 * K + 128 * K - 16,), (16, 600 * K, 16),
                                   (33 * 2048 * K + 1008,)])
def test_every_byte_arrives(host, sizes):  # noqa: F811
    engine = Engine(host)
    for seed in range(2):
        assert engine.fetch(*sizes, seed=seed) == (True, True)
    engine.close()
    assert host.fake_pinned() == 0 and host.fake_events() == 0
