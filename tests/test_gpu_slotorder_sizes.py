"""The device slot order where its kernels change hands: tables up to 8,192 slots (6,553 keys) run in one
workgroup, larger ones in launches of their own; the walk keys' order comes from the same epochs when
their sorted layout is not provably the slot order."""
import os

import numpy as np
import pytest

from conftest import run_oracle
from test_gpu_slotorder import clone_order, engine  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kept", [1, 5, 6, 7, 12, 13, 3276, 3277, 6552, 6553, 6554, 13107, 13108, 26215])
@pytest.mark.parametrize("transient", [0.0, 0.3])
def test_kept_counts_around_growths(engine, kept, transient):  # noqa: F811
    rnd = np.random.default_rng(kept)
    keys = rnd.permutation(np.arange(1000, 1100 + 2 * kept)).astype(np.int32)
    tr = (rnd.random(len(keys)) < transient).astype(np.uint8)
    # exactly `kept` keys stay; the last operation is the one that fills the table, or one after it
    end = int(np.nonzero(np.cumsum(tr == 0) == kept)[0][0]) + 1
    for n in (end, end + int(tr[end] == 1)):
        want, _ = clone_order(keys[:n], tr[:n])
        got = engine.slot_order(keys[:n], tr[:n])
        assert got is not None and got.tolist() == want


def test_walk_keys_whose_sorted_layout_is_not_the_order(tools, dataset):
    """200 kb of consecutive keys reach a displacement of 6 (the sorted layout then proves nothing)."""
    from rabbitvar_amd import read_fasta, read_rvb
    from rabbitvar_amd.engine import Engine

    d = dataset("c1")
    name, seq = read_fasta(os.path.join(d, "ref.fa"))
    want, _ = run_oracle(d, f"chrS:1-{len(seq)}", ["--fisher"], out="slot_sizes.txt")
    eng = Engine(sample="S1", fisher=1)
    got = eng.run_region(name, 1, len(seq), read_rvb(os.path.join(d, "reads.rvb")), name, seq)
    order = eng.stats()["order_sorted"]
    eng.close()
    assert got == want
    assert order == 7  # both orders came from the device


def test_order_ends_at_an_early_growth(tools, tmp_path):
    """-p keeps nearly every position, and they are inserted in another table's slot order: a small
    table's low homes crowd into one run that overflows.  The device's part ends there (a fraction of a
    millisecond; 7 ms when the later tables were still packed) and the host orders."""
    import subprocess

    from rabbitvar_amd import read_fasta, read_rvb
    from rabbitvar_amd.engine import Engine

    d = str(tmp_path)
    subprocess.run([tools["synth"], "--out", d, "--seed", "3", "--len", "24000", "--depth", "30"], check=True,
                   capture_output=True)
    name, seq = read_fasta(os.path.join(d, "ref.fa"))
    reads = read_rvb(os.path.join(d, "reads.rvb"))
    want, _ = run_oracle(d, f"{name}:2001-22000", ["-p"])
    eng = Engine(sample="S1", doPileup=1)
    ms = []
    for _ in range(5):
        assert eng.run_region(name, 2001, 22000, reads, name, seq) == want
        st = eng.stats()
        assert st["order_ops"] > 15000 and st["order_sorted"] == 3  # ordered on the host
        ms.append(st["order_device_ms"])
    eng.close()
    print("order on the device, ms:", ms, flush=True)
    assert min(ms) < 2.5
