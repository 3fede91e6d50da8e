"""GPU test of the memory that contexts keep of destroyed vectors: one bound for
all contexts of a device, almost nothing without vectors, all of it on trim."""
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20
SIXTEENTH = (288 << 30) // 16  # of MI355X's memory


def _vectors(dev, nbytes, count):
    from sep_code_amd.operator import DeviceVector
    return [DeviceVector(dev, nbytes // 4) for _ in range(count)]


def test_contexts_share_one_bound():
    """Two contexts that each destroy 14 GB of vectors keep a sixteenth of the
    device together, not each."""
    from sep_code_amd.device import BornDevice
    part = 7168 * MB
    with BornDevice(0) as a, BornDevice(0) as b:
        live = [v for d in (a, b) for v in _vectors(d, 1024, 1)]
        base = a.device_bytes() + b.device_bytes()
        for d in (a, b):
            for v in _vectors(d, part, 2):
                v.close()
        kept = a.device_bytes() + b.device_bytes() - base
        assert part <= kept <= SIXTEENTH
        # what a context may not keep is free for others
        for d in (a, b):
            d.trim()
        assert a.device_bytes() + b.device_bytes() == base
        for v in live:
            v.close()


def test_context_without_vectors_gives_its_memory_back():
    from sep_code_amd.device import BornDevice
    with BornDevice(0) as d:
        base = d.device_bytes()
        vs = _vectors(d, 1024 * MB, 3)
        vs[0].close()
        assert d.device_bytes() - base == 1024 * MB  # kept for the next
        for v in vs[1:]:
            v.close()
        assert d.device_bytes() - base <= 64 * MB


def test_trim_frees_while_vectors_live():
    from sep_code_amd.device import BornDevice
    with BornDevice(0) as d:
        live = _vectors(d, MB, 1)[0]
        for v in _vectors(d, 512 * MB, 2):
            v.close()
        held = d.device_bytes()
        d.trim()
        assert held - d.device_bytes() == 1024 * MB
        assert not live.numpy().any()
        live.close()
        with pytest.raises(Exception):
            d.close()
            d.trim()
