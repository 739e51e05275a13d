"""The device bytes that a server reports, and that its budget is held to, are
those it holds: per slot a descriptor (144 bytes), the geometry of a 512 x 512
grid (4096 doubles) and a y factor table (3120 reals), a list of 256 tiles of 24
bytes a slot with the slots' numbers behind it, and the arena's two grids.
"""
import pytest

import locvolcalib as lvc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [1, 7, 64])
@pytest.mark.parametrize("precision,real", [(lvc.PRECISION_FP32_REFINE, 4), (lvc.PRECISION_FP64, 8)])
def test_device_bytes(slots, precision, real):
    print(f"case: a server of {slots} slots, precision {precision}", flush=True)
    tables = slots * (144 + 8 * 4096 + real * 3120 + 24 * 256) + (4 * slots + 15) // 16 * 16
    grid = 2 * 64 * real  # the least extent, of R and of Y
    with lvc.LocVolCalib() as ctx:
        server = lvc.Server(ctx, max_slots=slots, precision=precision)
        assert server.device_bytes() == tables + slots * 2 * 512 * 512 * real
        server.free()
        server = lvc.Server(ctx, max_slots=slots, mem_budget=tables + grid, precision=precision)
        assert server.device_bytes() == tables + grid
        server.free()
        with pytest.raises(lvc.LocVolCalibError, match="does not cover"):
            lvc.Server(ctx, max_slots=slots, mem_budget=tables + grid - 1, precision=precision)
