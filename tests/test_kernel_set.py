"""The stage kernels that the library holds (its own symbols): one of the fused tile with 64-bit offsets per
basis and flux, since no mesh but a strip reaches it, and every tile shape of the 32-bit ones."""
import re
import subprocess


def _fused_tiles():
    import hyperboliconvergence_amd as hca
    out = subprocess.run(["nm", "-C", "--defined-only", hca.LIBPATH], capture_output=True, text=True, check=True).stdout
    # FusedTile<basis, flux, ti, tj, lanes, offset type, uniform, fold>
    return set(re.findall(r"k_stage<hc::FusedTile<(\d), (\d), (\d+), (\d+), (\d+), (unsigned [\w ]+), (\d), (\d)>", out))


def test_fused_kernels_by_offset_width():
    tiles = _fused_tiles()
    wide = [t for t in tiles if t[5] == "unsigned long long"]
    assert sorted(t[:2] for t in wide) == [(b, f) for b in "01" for f in "01456"]
    assert {t[2:5] for t in wide} == {("7", "16", "256")}
    narrow = [t for t in tiles if t[5] == "unsigned int"]
    assert len(narrow) == 2 * 5 * 3 * 2 * 2   # bases, fluxes, shapes, geometry, fold
