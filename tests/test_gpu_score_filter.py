"""Variants the output filter drops on their counts alone are not built; what they do to the later
variants of their position (the genotype they extend, the lookup that ends it) must stay.  Against
the oracle: indel-rich positions with many descriptors, insertions and deletions moved (-3), a filter
that drops nearly everything, and windows cut by the contig's ends."""
import os

import pytest

from conftest import run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("region", [None, (1, 400), (59600, 60000)])
@pytest.mark.parametrize("extra,options", [([], {}), (["-3"], {"moveIndelsTo3": 1}), (["-f", "0.2"], {"freq": 0.2}),
                                           (["-r", "1"], {"minr": 1})])
def test_filtered_variants(dataset, region, extra, options):
    from rabbitvar_amd import read_fasta, read_rvb
    from rabbitvar_amd.engine import Engine

    d = dataset("edge")
    name, seq = read_fasta(os.path.join(d, "ref.fa"))
    s, e = region or (1, len(seq))
    tag = "_".join(x.strip("-") for x in extra) or "plain"
    want, _ = run_oracle(d, f"chrS:{s}-{e}", ["--fisher"] + extra, out=f"filter_{tag}_{s}.txt")
    eng = Engine(sample="S1", fisher=1, **options)
    got = eng.run_region(name, s, e, read_rvb(os.path.join(d, "reads.rvb")).select(s, e), name, seq)
    eng.close()
    assert len(want.splitlines()) > (100 if region is None else 0)
    assert got == want
