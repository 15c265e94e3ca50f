"""The units of the library: a first launch loads the code of the whole unit
that its kernel is in, so each velocity set, stencil and precision has one of
its own, and kernels without a stencil among their parameters are local to
their unit (else one instance, in one of the units, would serve all)."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    'idea.deploy_amd', 'csrc')


def test_one_stencil_and_precision_per_unit():
    seen = []
    for f in sorted(glob.glob(os.path.join(CSRC, 'sc_*.hip'))):
        found = re.findall(r'ops_for_(f\d\d)<(D\w+), (D\dE\d)>', open(f).read())
        assert len(found) == 1, f
        seen += found
    assert len(set(seen)) == len(seen) == 12


def test_kernels_shared_by_units_are_local():
    src = open(os.path.join(CSRC, 'sc_kernels.h')).read()
    kernels = re.findall(r'template <([^>]*)>\n(static )?__global__[^\n]*\n(k_\w+)\(', src)
    assert len(kernels) == 13
    for params, local, name in kernels:
        assert bool(local) == ('class ES' not in params), name
