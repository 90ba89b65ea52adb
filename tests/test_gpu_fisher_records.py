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


@pytest.mark.parametrize("depth,options", [(60, {"freq": 0.0, "minr": 1}), (4000, {"freq": 0.0, "minr": 1}), (60, {"doPileup": 1})])
def test_same_bits_as_the_serial_test(tools, tmp_path, depth, options):
    """Each record's p-value, summed by a wavefront, has the bits of the same table's serial sum (a lane
    alone, through rv_debug_fisher): shallow and deep records, and the near-certain ones -p prints."""
    import numpy as np

    from rabbitvar_amd import read_fasta, read_rvb
    from rabbitvar_amd.engine import Engine

    d = str(tmp_path)
    subprocess.run([tools["synth"], "--out", d, "--seed", "3", "--len", "6000", "--depth", str(depth), "--snv-rate", "0.02",
                    "--indel-rate", "0.002"], check=True, capture_output=True)
    name, seq = read_fasta(os.path.join(d, "ref.fa"))
    eng = Engine(sample="S1", fisher=1, **options)
    _, calls = eng.run_region_calls(name, 1001, 5000, read_rvb(os.path.join(d, "reads.rvb")), name, seq)
    tables = np.array([[c[k] for k in ("ref_fwd", "ref_rev", "var_fwd", "var_rev")] for c in calls])
    serial = eng.fisher(tables)[:, 0]
    eng.close()
    wave = np.array([c["fisher_p"] for c in calls])
    print(f"{len(calls)} records, totals up to {tables.sum(axis=1).max()}, {len(np.unique(wave))} values", flush=True)
    assert len(calls) > 300 and len(np.unique(wave)) > 50
    assert np.array_equal(wave.view(np.int64), serial.view(np.int64))


def test_text_overflow_then_retry(tools, tmp_path):
    """More allele text than the first pass has room for (60 different 100-base insertions at each of
    900 positions; 160 bytes a record are set aside, for 65,536 records, 8 a record-list position and
    one a 16 positions): that pass's slots are not all written, and the repeated one prints the
    oracle's lines."""
    import random

    from rabbitvar_amd import batch_from_records, write_rvb
    from rabbitvar_amd.engine import Engine

    rnd = random.Random(4)
    npos, alleles, step, size = 900, 60, 12, 100
    ref = "".join(rnd.choices("ACGT", k=2000 + npos * step))
    recs = []
    for i in range(npos):
        p = 500 + i * step
        for k in range(alleles):
            seq = ref[p:p + 30] + "".join(rnd.choices("ACGT", k=size)) + ref[p + 30:p + 60]
            recs.append({"pos0": p, "flag": 16 if k % 2 else 0, "mapq": 60, "nm": size, "seq": seq, "qual": [30] * len(seq),
                         "cigar": [(0, 30), (1, size), (0, 30)]})
    batch = batch_from_records(recs)
    d, s, e = str(tmp_path), 400, len(ref) - 600
    with open(os.path.join(d, "ref.fa"), "w") as f:
        f.write(">chrS\n" + ref + "\n")
    write_rvb(os.path.join(d, "reads.rvb"), batch)
    want, _ = run_oracle(d, f"chrS:{s}-{e}", ["--fisher", "-k", "0", "-f", "0.0001", "-r", "1"])
    lines = want.splitlines()
    # the allele and the descriptor of an insertion, and the two flanks
    text = sum(2 * len(ln.split("\t")[6]) + 40 for ln in lines)
    assert len(lines) < 65536 and text > 160 * (65536 + 8 * npos + (e - s + 4000) // 16)
    bases = ref.encode()
    eng = Engine(sample="S1", fisher=1, performLocalRealignment=0, freq=0.0001, minr=1)
    got = eng.run_region("chrS", s, e, batch, "chrS", bases)
    again = eng.run_region("chrS", s, e, batch, "chrS", bases)
    eng.close()
    assert got == want and again == want
