"""The modified enumeration for every number of modable acids that a database packs, bit by bit
against the oracle's."""
import pytest

import test_gpu_mods

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("acids", ["M", "CM", "MST", "KMST", "KMSTY", "KMNSTY", "KMNQSTY"])
def test_enumeration_for_any_number_of_acids(orc, acids):
    from hfx_amd import pipeline, synth

    prot = synth.make_proteins(300, seed=81)
    mass = orc.mass_table()
    r, tc, tn = orc.digest(prot.seq, prot.seg, mass, rule=1, missed=1, p_rule=1, min_len=7, max_len=30)
    sp = synth.make_spectra(prot, r, tc, tn, 12, seed=82, charges=(1, 2, 3, 4))
    ctx, mi = pipeline.Ctx(0), pipeline.mod_info({a: 9.5 + 8 * k for k, a in enumerate(acids)}, 4)
    assert mi.num_ma == len(acids)
    db = pipeline.DeviceDB(pipeline.HostDB(prot.seq, r, tc, tn, mass), ma=mi.ma)
    dsp = pipeline.DeviceSpectra(ctx, sp.pcr, sp.charge, sp.mz, sp.inten, sp.off, test_gpu_mods.STRIDE)
    res = pipeline.ModSearch(ctx, db, dsp, mi, eps=3.0, topn=5).run()
    test_gpu_mods.test_enumeration_bit_exact(
        dict(prot=prot, r=r, tc=tc, tn=tn, mi=mi, db=db, dsp=dsp, res=res), orc)
