"""Counts at which the kernels' rounds end, against the oracle: signals of as
many events as a block takes in one round (256 threads, four rounds in flight)
and one less or more, tiles of 64, 256 and 1,024 words (the copy of a tile's
entries takes 64 accesses of four, four of them in flight), and tiles handed
out to so few workgroups that only some of the ticket counters are used."""
import re
import sys

import pytest

import gls
import oracle_bind

pytestmark = pytest.mark.gpu

LENGTHS = (1, 3, 255, 256, 257, 1023, 1024, 1025, 4097)


@pytest.fixture(scope="module")
def ctx():
    c = gls.Context(0)
    yield c
    c.close()


def cut_vcd(src, dst):
    """Keeps the first LENGTHS[k] changes of the k-th signal."""
    head, body = open(src).read().split("$enddefinitions $end\n")
    left, out = {}, []
    for tok in body.split():
        if tok[0] in "01xzXZ":
            sig = tok[1:]
            if sig not in left:
                left[sig] = LENGTHS[len(left) % len(LENGTHS)]
            left[sig] -= 1
            if left[sig] < 0:
                continue
        out.append(tok)
    with open(dst, "w") as f:
        f.write(head + "$enddefinitions $end\n" + "\n".join(out) + "\n")


@pytest.fixture(scope="module")
def case(tmp_path_factory):
    t = str(tmp_path_factory.mktemp("edges"))
    d = gls.Design.generate(3, 811, 60, 3, len(LENGTHS))
    paths = [t + "/" + n for n in ("lib.vlib", "n.gv", "n.sdf", "s.vcd")]
    d.write(*paths[:3])
    gls.Stimulus.generate(d, 812, 60000, 10.0, 0.05).write_vcd(t + "/all.vcd")
    cut_vcd(t + "/all.vcd", paths[3])
    window = (7001, 59000)
    return d, gls.Stimulus.from_vcd(paths[3]), window, oracle_bind.run(*paths, *window, t)


def toggles(wave, on, off):
    return sum(1 for (_, p), (t, v) in zip(wave, wave[1:]) if {p, v} == {0, 3} and on < t <= off)


def check(r, want, what):
    assert r.stats()["n_events"] == want["n_events"], what
    assert r.waves_hash() == want["waves_hash"], what
    assert re.sub(r" \(TC \d+\)", "", r.saif_text()) == want["saif"], what


@pytest.mark.parametrize("seg,chunk", [(0, 0), (1, 0), (4, 0), (16, 0), (16, 17011)])
def test_round_ends(ctx, case, seg, chunk):
    print("round ends", seg, chunk, flush=True)
    sys.stdout.flush()
    d, s, (on, off), want = case
    r = ctx.simulate(d, s, on, off, keep_waves=True, saif_tc=True, seg_events=seg, chunk_ps=chunk)
    check(r, want, (seg, chunk))
    names = re.findall(r"^      \((\S+)\n         \(T0", r.saif_text(), re.M)
    assert len(names) > 20
    for net in names:
        assert r.net_toggles(net) == toggles(r.waveform(net), on, off), net
    r.close()


@pytest.mark.parametrize("blocks", [1, 7, 8, 9, 17, 25, 40])
def test_few_workgroups(ctx, case, blocks):
    print("workgroups", blocks, flush=True)
    sys.stdout.flush()
    d, s, (on, off), want = case
    r = ctx.simulate(d, s, on, off, keep_waves=True, seg_events=1, level_blocks=blocks)
    assert r.stats()["tiles"] > 8 * blocks
    check(r, want, blocks)
    r.close()


@pytest.mark.parametrize("burst", [900, 1400, 1700, 2900, 3400, 5000])
def test_tiles_too_long_for_lds(ctx, burst, tmp_path):
    """Half of the signals change all along, the others `burst` times in a short
    stretch: at one word a lane its tiles hold more than LDS does, with their
    stacks (about 1,500 words) or without them (about 3,000)."""
    print("too long", burst, flush=True)
    sys.stdout.flush()
    t = str(tmp_path)
    d = gls.Design.generate(3, 813, 40, 2, 8)
    paths = [t + "/" + n for n in ("lib.vlib", "n.gv", "n.sdf", "s.vcd")]
    d.write(*paths[:3])
    gls.Stimulus.generate(d, 814, 1000, 10.0, 0.05).write_vcd(t + "/all.vcd")
    head, body = open(t + "/all.vcd").read().split("$enddefinitions $end\n")
    events = []
    for k, sig in enumerate(sorted({tok[1:] for tok in body.split() if tok[0] in "01xzXZ"})):
        n, at, gap = (1100, 10 + k, 50) if k % 2 == 0 else (burst, 20000 + k, 3)
        events += [(at + gap * i, sig, "01"[(i + k) & 1]) for i in range(n)]
    events.sort()
    with open(paths[3], "w") as f:
        f.write(head + "$enddefinitions $end\n")
        for at, sig, v in events:
            f.write("#%d\n%s%s\n" % (at, v, sig))
    s = gls.Stimulus.from_vcd(paths[3])
    want = oracle_bind.run(*paths, 100, 60000, t)
    r = ctx.simulate(d, s, 100, 60000, keep_waves=True, seg_events=1)
    assert r.stats()["tiles_hbm"] > 0 or burst < 1500
    check(r, want, burst)
    r.close()


@pytest.mark.parametrize("workers,max_batch", [(1, 4), (3, 4), (4, 1)])
def test_jobs_that_find_a_free_worker_run_alone(ctx, workers, max_batch):
    """Every job's results are its own run's; the first jobs, one a worker, run
    by themselves however fast they are submitted, so that their counts too are
    those of a run of their own."""
    print("workers", workers, max_batch, flush=True)
    sys.stdout.flush()
    d = gls.Design.generate(1, 815, 900, 12, 20)
    ss = [gls.Stimulus.generate(d, 820 + i, 40000, 150.0, 0.02) for i in range(7)]
    alone = []
    for s in ss:
        r = ctx.simulate(d, s, 0, 40001)
        alone.append((r.saif_text(), r.stats()["n_events"]))
        r.close()
    srv = gls.Server(ctx, max_running=workers, max_batch=max_batch)
    for _ in range(3):
        jobs = [srv.submit(d, s, 0, 40001) for s in ss]
        for i, j in enumerate(jobs):
            assert srv.wait(j) == 0
            assert srv.saif_text(j) == alone[i][0], i
            if i < workers:
                assert srv.info(j)["n_events"] == alone[i][1], i
    srv.close()
