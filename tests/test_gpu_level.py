"""Where tiles begin: the search for a boundary's words in every input guesses
from how far the boundary lies inside the leader's words.  Inputs whose events
follow time evenly, lie in one short burst, only at one end, or are one word
long, against the oracle; gates of one tile and of hundreds, levels of more
gates than one plan block holds."""
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


def warp_vcd(src, dst, t_end):
    """Moves each signal's events: evenly (as they are), into a burst in the
    middle, to the first or last hundredth, or all but the first away."""
    head, body = open(src).read().split("$enddefinitions $end\n")
    ids, last, events, t = {}, {}, [], 0
    for tok in body.split():
        if tok[0] == "#":
            t = int(tok[1:])
        elif tok[0] in "01xzXZ":
            sig = tok[1:]
            k = ids.setdefault(sig, len(ids)) % 5
            at = (t, t_end // 2 + t // 100, t // 100, t_end - t_end // 100 + t // 100, t)[k]
            if k == 4 and sig in last:
                continue
            last[sig] = max(at, last.get(sig, -1) + 1)  # one event of a signal a time
            events.append((last[sig], sig, tok))
    events.sort(key=lambda e: e[0])
    with open(dst, "w") as f:
        f.write(head + "$enddefinitions $end\n")
        now = -1
        for at, _, tok in events:
            if at != now:
                f.write("#%d\n" % at)
                now = at
            f.write(tok + "\n")


@pytest.mark.parametrize("seed,cells,levels,t_end,gap", [(1, 60, 3, 200000, 60.0), (2, 1100, 2, 9000, 45.0),
                                                         (3, 20, 5, 400, 8.0)])
def test_tile_boundaries_of_uneven_inputs(ctx, seed, cells, levels, t_end, gap, tmp_path):
    print("boundaries", seed, cells, levels, flush=True)
    sys.stdout.flush()
    d = gls.Design.generate(3, 500 + seed, cells, levels, 10)
    paths = [str(tmp_path / n) for n in ("lib.vlib", "n.gv", "n.sdf", "s.vcd")]
    d.write(*paths[:3])
    s = gls.Stimulus.generate(d, 60 + seed, t_end, gap, 0.05)
    s.write_vcd(str(tmp_path / "even.vcd"))
    warp_vcd(str(tmp_path / "even.vcd"), paths[3], t_end)
    s = gls.Stimulus.from_vcd(paths[3])
    start, end = t_end // 7, t_end + 100
    want = oracle_bind.run(*paths, start, end, str(tmp_path))
    for seg in (0, 1, 3):
        r = ctx.simulate(d, s, start, end, keep_waves=True, seg_events=seg)
        assert r.stats()["n_events"] == want["n_events"], seg
        assert r.waves_hash() == want["waves_hash"], seg
        assert r.saif_text() == want["saif"], seg
        r.close()


@pytest.mark.parametrize("cells,t_end,gap", [(12, 40000, 20.0), (300, 30000, 40.0)])
def test_lane_shares_of_small_levels(ctx, cells, t_end, gap, tmp_path):
    """The default lane share depends on how many workgroups a level has to
    fill (16 to 32 words); any share gives the same waveforms, and in a batch
    it stays fixed."""
    print("shares", cells, flush=True)
    sys.stdout.flush()
    d = gls.Design.generate(3, 700 + cells, cells, 4, 8)
    paths = [str(tmp_path / n) for n in ("lib.vlib", "n.gv", "n.sdf", "s.vcd")]
    d.write(*paths[:3])
    s = gls.Stimulus.generate(d, 71, t_end, gap, 0.05)
    s.write_vcd(paths[3])
    want = oracle_bind.run(*paths, 0, t_end, str(tmp_path))
    tiles = []
    for blocks in (1, 8, 64, 0):
        r = ctx.simulate(d, s, 0, t_end, keep_waves=True, level_blocks=blocks)
        assert r.stats()["n_events"] == want["n_events"], blocks
        assert r.waves_hash() == want["waves_hash"], blocks
        assert r.saif_text() == want["saif"], blocks
        tiles.append(r.stats()["tiles"])
        r.close()
    assert tiles[0] <= tiles[1] <= tiles[2] <= tiles[3] and tiles[0] < tiles[3]
    run = ctx.prepare_batch([d, d], [s, s], [0, 0], [t_end, t_end])
    run.execute()
    assert run.stats()["tiles"] == 2 * tiles[0]
    assert run.instance_saif_text(1) == want["saif"]
    run.close()
