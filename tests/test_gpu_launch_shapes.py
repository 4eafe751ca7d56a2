"""Every launch shape that acts on a class gives the same bits: the band
solver's in the mixed class that still has two, the SAB/DAB kernel's in the
mixed classes of the symmetric path."""
import pytest

from aeroapps_amd import tune as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nstreams,acts", [(8, (True, True)), (6, (False, True)), (3, (False, True))])
def test_acting_shapes_bit_identical(gpu, nstreams, acts):
    import torch
    print(f"case acting shapes N={nstreams}", flush=True)
    assert T.live(nstreams, 1, 1) == acts
    res = T.tune_class(torch, nstreams, 1, (1,), ncol=300, reps=1, log=lambda m: None)   # raises where bits differ
    best, times = res[1]
    assert best in times and len(set(times.values())) > 1
