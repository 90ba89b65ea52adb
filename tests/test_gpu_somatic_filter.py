"""Somatic pairs under filters that change which positions can print (a position is emitted only when
one of its variants passes the count checks in either sample): against the oracle, text for text."""
import pytest

from test_gpu_somatic import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra,options", [(["-f", "0.2"], {"freq": 0.2}), (["-f", "0"], {"freq": 0.0}),
                                           (["-r", "1"], {"minr": 1}), (["-r", "9"], {"minr": 9})])
@pytest.mark.parametrize("start,end", [(1, 12000), (59000, 60000)])
def test_somatic_filters(dataset, start, end, extra, options):
    got, want = _run(dataset("som_edge"), start, end, ["--fisher"] + extra, f"som_f_{''.join(extra)}_{start}.txt", fisher=1,
                     **options)
    assert want.count("\n") >= (76 if end == 12000 else 4)
    assert got == want
