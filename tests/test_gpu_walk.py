"""The forms of the walk's tables (fan-in 1..6, delays that depend on an
input's edge or not) and its lane shares at tile edges, against the oracle.

Designs of the generator's full library with some IOPATHs rewritten into
posedge / negedge pairs, a posedge record alone, or an edge record beside an
edge-independent one: every fan-in then occurs with and without edge-dependent
delays.  Tile sizes from one word a lane to more than LDS holds, one time chunk
and many."""
import random
import re
import sys

import pytest

import gls
import oracle_bind

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = gls.Context(0)
    yield c
    c.close()


def with_edges(sdf, rng):
    def one(m):
        pad, pin, rest = m.group(1), m.group(2), m.group(3)

        def delays():
            a, b = rng.randint(1, 60), rng.randint(1, 60)
            return "(%d:%d:%d) (%d:%d:%d)" % (a, a, a, b, b, b)
        k = rng.randrange(6)
        if k == 0:
            return "%s(IOPATH (posedge %s) %s %s)\n%s(IOPATH (negedge %s) %s %s)" % (
                pad, pin, rest, delays(), pad, pin, rest, delays())
        if k == 1:
            return "%s(IOPATH (posedge %s) %s %s)" % (pad, pin, rest, delays())
        if k == 2:
            return m.group(0) + "\n%s(IOPATH (negedge %s) %s %s)" % (pad, pin, rest, delays())
        return m.group(0)
    return re.sub(r"^( *)\(IOPATH (\w+) (\w+) \([^\n]*$", one, sdf, flags=re.M)


@pytest.mark.parametrize("seed,cells,t_end,gap", [(1, 90, 30000, 60.0), (2, 150, 9000, 12.0),
                                                  (3, 60, 200000, 300.0), (4, 40, 700, 4.0)])
def test_table_forms_against_oracle(ctx, seed, cells, t_end, gap, tmp_path):
    print("walk", seed, cells, t_end, gap, flush=True)
    sys.stdout.flush()
    rng = random.Random(seed)
    d = gls.Design.generate(3, 9000 + seed, cells, 5, 9)
    paths = [str(tmp_path / n) for n in ("lib.vlib", "n.gv", "n.sdf", "s.vcd")]
    d.write(*paths[:3])
    text = with_edges(open(paths[2]).read(), rng)
    open(paths[2], "w").write(text)
    d = gls.Design.from_files(*paths[:3])
    s = gls.Stimulus.generate(d, 40 + seed, t_end, gap, 0.05)
    s.write_vcd(paths[3])
    start, end = t_end // 5, t_end + 100
    want = oracle_bind.run(*paths, start, end, str(tmp_path))
    for seg, chunk in ((0, 0), (1, 0), (2, 0), (3, t_end // 3), (31, 0), (33, 211), (1 << 20, 0)):
        r = ctx.simulate(d, s, start, end, keep_waves=True, seg_events=seg, chunk_ps=chunk)
        assert r.stats()["n_events"] == want["n_events"], (seg, chunk)
        assert r.waves_hash() == want["waves_hash"], (seg, chunk)
        assert r.saif_text() == want["saif"], (seg, chunk)
        r.close()
