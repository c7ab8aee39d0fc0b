"""What the benchmark's line says about the kernels that ran: the unions walked
and the bytes staged, from the entry points launched and the unions' entries."""
import pytest

import bench

D, LENS = 128, 900
TILE = 2 * 64 * D * 2  # K and V


@pytest.mark.parametrize("launched,quad,forward,dq", [
    ({"prism_bsa_fwd_either", "prism_bsa_bwd_dkdv", "prism_bsa_bwd_dq"}, 400, "quad", "pair"),
    ({"prism_bsa_fwd_either", "prism_bsa_bwd_dkdv", "prism_bsa_bwd_dq_quad"}, 401, "pair", "quad"),
    ({"prism_bsa_fwd", "prism_bsa_bwd_dkdv_split", "prism_bsa_bwd_dq_split"}, None, "pair", "split pair"),
    ({"prism_bsa_fwd_tile"}, None, "tile", None)], ids=str)
def test_walked_unions_and_staged_bytes(launched, quad, forward, dq):
    entries = {"pair": 600, "quad": quad, "key": 700}
    walked = bench.walked_unions(launched, entries)
    assert walked == {"forward": forward, "dq": dq}
    staged = bench.staged_tile_bytes(entries, walked, LENS, D)
    count = {"pair": 600, "split pair": 600, "quad": quad, "tile": LENS}
    for name in launched:
        want = (TILE + 512) * 700 if "dkdv" in name else TILE * count[forward if "fwd" in name else dq]
        assert staged[name] == want, name
    slots = bench.slot_efficiency(entries, walked, LENS)
    assert slots["query_unions"] == walked and slots["union_slot_efficiency"] == 0.75
    assert slots["quad_union_slot_efficiency"] == (None if quad is None else round(LENS / (4 * quad), 4))
