"""The SAIF report of a netlist large enough for several writer threads, rebuilt
record by record from the per-net counters; the size query and a buffer that is
one byte short."""
import ctypes
import re

import pytest

import gls

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,with_tc", [(50, False), (8100, False), (12345, True)])
def test_report_equals_the_counters(cells, with_tc, tmp_path):
    print("saif", cells, with_tc, flush=True)
    ctx = gls.Context(0)
    d = gls.Design.generate(1, 4100 + cells, cells, 6, 20)
    s = gls.Stimulus.generate(d, 5, 3000, 300.0, 0.02)
    r = ctx.simulate(d, s, 10, 2990, saif_tc=with_tc)
    text = r.saif_text()
    names = re.findall(r"^      \((\S+)\n", text, re.M)
    assert len(names) == cells + 20 and names == sorted(names)
    want = "(TIMESCALE 1 ps)\n(DURATION 2980)\n(INSTANCE root\n   (NET\n"
    for n in names:
        want += "      (%s\n         (T0 %d) (T1 %d) (TX %d)" % ((n,) + r.net_saif(n))
        want += " (TC %d)" % r.net_toggles(n) if with_tc else ""
        want += "\n      )\n"
    assert text == want + "   )\n\n)\n"
    path = str(tmp_path / "out.saif")
    r.write_saif(path)
    assert open(path).read() == text
    n = ctypes.c_size_t()
    buf = ctypes.create_string_buffer(len(text))
    assert gls.load().gls_run_saif_text(r.ptr, buf, len(text) - 1, ctypes.byref(n)) == -1
    assert n.value == len(text)
    r.close()
    ctx.close()
