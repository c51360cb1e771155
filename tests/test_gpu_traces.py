"""The sampled traces of a region at the sizes where their log and replay change.

A trace's domains go to a log of runs that is read 64 entries at a time and
holds all 200 traces of a region only from about M = 150 on; below, several
passes fill it in turn. Covered: one-node, smallest and one-pass models, M at
the edges of 4 striped lanes and of 64 cells (the region's Forward holds up to
eight per lane, M = 512, in registers), regions of one residue, around 64 residues
and of several domains, and 1, 3 and 200 traces. The sampled domains and the
clusters equal the oracle's exactly; the residues' null2 scores differ by logf's
last bit per residue (1e-6 nats, as for the regions of whole searches).
"""
import numpy as np
import pytest

import oracle
from biobench2_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 4, 5, 32, 33, 63, 64, 65, 128, 129, 149, 160, 256, 257, 384, 385, 400, 512, 513, 700])
def test_traces_equal_the_oracle_at_log_and_region_edges(gpu, tmp_path, M):
    rng = np.random.default_rng([11, M])
    h = synth.random_profile(M, rng, f"traces_M{M}")
    h.stats = (-9.0, 0.6931, -9.5, 0.6931, -5.0, 0.6931)
    path = str(tmp_path / "traces.hmm")
    synth.write_hmm(path, [h])
    om = gpu.OProfile.from_file(path)
    hh = synth.read_hmm_probs(path)
    regs = [synth.iid_residues(L, rng) for L in (1, 2, 63, 64, 65)]
    regs.append(np.concatenate([x for c in synth.emit_homologs(hh, 3, rng) for x in (c, synth.iid_residues(3, rng))])
                .astype(np.uint8))
    for reg in regs:
        om.reconfig_length(reg.size + 50)
        t = om.tables()
        for ns in ((1, 3, 200) if reg.size > 1 else (200,)):
            st, cl, n2, segs = oracle.region_multidomain(reg, t, 1, reg.size, nsamples=ns, want_segs=True)
            assert st == 0
            g = gpu.region_trace_ensemble(reg, reg.size + 50, om, nsamples=ns, matrix=True)
            assert g["nseg"] == len(segs) and np.array_equal(segs, g["segs"]), (reg.size, ns)
            assert g["clusters"] == cl, (reg.size, ns)
            assert float(np.max(np.abs(n2 - g["n2sc"]))) <= 1e-6, (reg.size, ns)
