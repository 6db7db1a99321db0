"""The encoder refuses a step whose memory lies beyond the 32-bit word offsets
of its dispatches, before it allocates the fields."""
import pytest

import te_host


@pytest.mark.parametrize("kw", [dict(nx=1200, ny=1200, nz=60), dict(nx=40000, ny=400, nz=8, open_x=1, open_y=1)])
def test_a_step_beyond_32_bit_offsets_is_refused(kw):
    with pytest.raises(te_host.TeError, match="2\\^32 words"):
        te_host.Run(te_host.config(tke=1, dz=300.0, **kw), encode_only=True)
