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


@pytest.mark.parametrize("length,most_ms", [(12000, None), (30000, None), (200000, 0.6)])
def test_printed_positions_few_and_many(tools, tmp_path, length, most_ms):
    """Every mismatch prints: positions scored a wavefront each, near the 3,072 of them from which on they
    are scored a lane each, and far beyond, where a wavefront each took 0.93 ms of scoring."""
    import subprocess

    from rabbitvar_amd import read_fasta, read_rvb
    from rabbitvar_amd.engine import Engine

    d = str(tmp_path)
    subprocess.run([tools["synth"], "--out", d, "--seed", "3", "--len", str(length), "--depth", "60"], check=True,
                   capture_output=True)
    name, seq = read_fasta(os.path.join(d, "ref.fa"))
    s, e = 1001, length - 1000
    want, _ = run_oracle(d, f"{name}:{s}-{e}", ["--fisher", "-f", "0", "-r", "1"])
    reads = read_rvb(os.path.join(d, "reads.rvb"))
    eng = Engine(sample="S1", fisher=1, freq=0.0, minr=1)
    ms = []
    for _ in range(4):
        assert eng.run_region(name, s, e, reads, name, seq) == want
        ms.append(eng.stats()["score_ms"])
    eng.close()
    print(f"{want.count(chr(10))} lines, scoring ms {ms}", flush=True)
    assert most_ms is None or min(ms) < most_ms
