"""The Fisher column of the printed records, whose tails a wavefront sums in stretches of eleven terms,
64 stretches at a time: depths on both sides of one stretch and one batch, against the oracle's text."""
import os
import subprocess

import pytest

from conftest import run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth,extra,options", [(8, [], {}), (90, [], {}), (1500, [], {}), (4000, ["-p"], {"doPileup": 1})])
def test_fisher_column(tools, tmp_path, depth, extra, options):
    from rabbitvar_amd import read_fasta, read_rvb
    from rabbitvar_amd.engine import Engine

    d = str(tmp_path)
    subprocess.run([tools["synth"], "--out", d, "--seed", "3", "--len", "2500", "--depth", str(depth), "--snv-rate", "0.02",
                    "--indel-rate", "0.002"], check=True, capture_output=True)
    name, seq = read_fasta(os.path.join(d, "ref.fa"))
    s, e = (600, 1100) if extra else (300, 2200)
    want, _ = run_oracle(d, f"{name}:{s}-{e}", ["--fisher"] + extra)
    eng = Engine(sample="S1", fisher=1, **options)
    got = eng.run_region(name, s, e, read_rvb(os.path.join(d, "reads.rvb")).select(s, e), name, seq)
    eng.close()
    assert len(want.splitlines()) > 10
    assert got == want
