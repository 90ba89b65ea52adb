"""Reads of every length and shape where the pileup's steps change path, against the oracle: lengths at
the edges of a word, a wavefront and the staged copy; mismatches alone, in pairs and apart by the
multi-base reach, at the ends and at every 64th base; low qualities, N and IUPAC codes;
reads cut by the contig's ends; clips, indels and the rewritten ends of single M runs.  Whole numbers
and text: compared exactly."""
import os
import random

import pytest

from conftest import run_oracle

pytestmark = pytest.mark.gpu

L = 4000


def _build(d):
    from rabbitvar_amd import batch_from_records, write_rvb

    rnd = random.Random(11)
    s = [rnd.choice("ACGT") for _ in range(L)]
    s[300:304] = list("RNNY")
    s = "".join(s)
    os.makedirs(d, exist_ok=True)
    with open(os.path.join(d, "ref.fa"), "w") as f:
        f.write(">chrT\n" + "\n".join(s[i:i + 60] for i in range(0, L, 60)) + "\n")
    lens = [2, 3, 7, 8, 9, 10, 11, 15, 16, 17, 40, 63, 64, 65, 66, 100, 127, 128, 129, 150, 511, 512, 513, 700]
    recs = []

    def other(c):
        return rnd.choice([x for x in "ACGT" if x != c])

    for k in range(900):
        n = rnd.choice(lens)
        pos0 = 0 if k % 60 == 0 else L - n if k % 60 == 1 else rnd.randrange(0, L - n - 40)
        kind = rnd.randrange(6) if n >= 40 and k % 60 > 1 else 0
        cigar, seq = [(0, n)], s[pos0:pos0 + n]
        if kind == 1:
            a, b = rnd.choice([0, 3, 12]), rnd.choice([2, 14])
            cigar = ([(4, a)] if a else []) + [(0, n - a - b), (4, b)]
            seq = "".join(rnd.choice("ACGT") for _ in range(a)) + s[pos0:pos0 + n - a - b] + s[-b:]
        elif kind == 2:
            x, w = rnd.randrange(12, n - 12), rnd.choice([1, 2, 9])
            cigar, seq = [(0, x), (2, w), (0, n - x)], s[pos0:pos0 + x] + s[pos0 + x + w:pos0 + n + w]
        elif kind == 3:
            x, w = rnd.randrange(12, n - 20), rnd.choice([1, 3])
            cigar, seq = [(0, x), (1, w), (0, n - x - w)], s[pos0:pos0 + x] + "GT" * w + s[pos0 + x:pos0 + n]
            seq = seq[:x + w] + s[pos0 + x:pos0 + n - w]
        seq = list(seq)
        # mismatches: one, two side by side, two apart, near the ends, at a wavefront's edge
        at = set()
        for _ in range(rnd.randrange(4) if n > 8 else 0):  # (a shorter record has no room for two new clips)
            i = rnd.choice([0, 1, 2, n - 1, n - 2, n - 3, 62, 63, 64, 65, rnd.randrange(n)])
            at |= {j for j in rnd.choice([(i,), (i, i + 1), (i, i + 2), (i, i + 3), (i, i + 4)]) if 0 <= j < n}
        for i in at:
            seq[i] = other(seq[i])
        for i in range(n):
            if n > 8 and rnd.random() < 0.004:
                seq[i] = rnd.choice("NNR")
        qual = [rnd.choice([37, 37, 37, 30, 26, 22, 12]) if rnd.random() < 0.2 else 37 for _ in range(n)]
        if k % 17 == 0:
            qual[rnd.randrange(n)] = 1
        idlen = sum(w for op, w in cigar if op in (1, 2))
        recs.append({"pos0": pos0, "flag": 16 * (k % 2), "mapq": rnd.choice([60, 60, 20]), "nm": len(at) % 5 + idlen,
                     "seq": "".join(seq), "qual": qual, "cigar": cigar})
    recs.sort(key=lambda r: r["pos0"])
    write_rvb(os.path.join(d, "reads.rvb"), batch_from_records(recs))


OPTIONS = [([], {}), (["-q", "30.5"], {"goodq": 30.5}), (["-X", "5"], {"vext": 5}), (["-T", "50"], {"trimBasesAfter": 50}),
           (["-k", "0"], {"performLocalRealignment": 0})]


@pytest.mark.parametrize("region", [(1, L), (1, 1), (64, 700), (L - 90, L)])
@pytest.mark.parametrize("extra,options", OPTIONS)
def test_read_shapes(tools, tmp_path, region, extra, options):
    from rabbitvar_amd import read_fasta, read_rvb
    from rabbitvar_amd.engine import Engine

    d = str(tmp_path / "shapes")
    _build(d)
    name, seq = read_fasta(os.path.join(d, "ref.fa"))
    s, e = region
    want, want_dump = run_oracle(d, f"chrT:{s}-{e}", ["--fisher"] + extra, dump="pile.txt")
    reads = read_rvb(os.path.join(d, "reads.rvb")).select(s, e)
    eng = Engine(sample="S1", fisher=1, **options)
    dump = eng.debug_pileup(name, s, e, reads, name, seq)
    got = eng.run_region(name, s, e, reads, name, seq)
    eng.close()
    assert sorted(dump.splitlines()) == sorted(want_dump.splitlines())
    assert len(want_dump.splitlines()) > (1000 if region == (1, L) else 0)
    assert got == want


@pytest.mark.parametrize("realign,most_ms", [(1, 1.45), (0, 0.35)])
def test_an_indel_in_nearly_every_read(tools, tmp_path, realign, most_ms):
    """The CIGAR rewrite when nearly every read takes its rules: the oracle's lines, and a prep pass no
    slower than a lane per read (1.60 ms here with local realignment, 0.22 without)."""
    import subprocess

    from rabbitvar_amd import read_fasta, read_rvb
    from rabbitvar_amd.engine import Engine

    d = str(tmp_path)
    subprocess.run([tools["synth"], "--out", d, "--seed", "3", "--len", "300000", "--depth", "60", "--indel-rate", "0.02",
                    "--indel-max", "10"], check=True, capture_output=True)
    name, seq = read_fasta(os.path.join(d, "ref.fa"))
    want, _ = run_oracle(d, f"{name}:1001-299000", ["--fisher", "-k", str(realign)])
    reads = read_rvb(os.path.join(d, "reads.rvb"))
    eng = Engine(sample="S1", fisher=1, performLocalRealignment=realign)
    ms = []
    for _ in range(5):
        assert eng.run_region(name, 1001, 299000, reads, name, seq) == want
        ms.append(eng.stats()["prep_ms"])
    eng.close()
    print("prep ms:", ms, flush=True)
    assert want.count("\n") > 5000 and min(ms) < most_ms
