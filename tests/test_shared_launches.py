"""Launches of a region that do not depend on one another run as one: what shares, what never does, values under the
oracle, replays, the static scratch area."""
import re

import numpy as np
import pytest

from adhip import ir as IR, workloads as W
from adhip.device import lower_describe
from oracle.interp import OracleDevice


def _plan(build):
    proc, deps = build(OracleDevice()).finish()
    return lower_describe(proc, deps)


def _mlp(dev, batch=64, dims=(32, 64, 48, 8), iters=3, seed=1):
    return W.mlp_train(dev, batch, dims, iters, seed=seed)


def _sets(text):
    """The member launches of every shared launch, by label."""
    sets, lines = [], text.splitlines()
    for i, line in enumerate(lines):
        m = re.match(r"\s*shared\d+_(\d+)x, one launch", line)
        if m:
            sets.append([re.match(r"\s*launch (\S+)", lines[i + 1 + j]).group(1) for j in range(int(m.group(1)))])
    return sets


def test_what_does_not_depend_shares_a_launch():
    sets = _sets(_plan(_mlp))
    assert sum(map(len, sets)) - len(sets) >= 8, sets   # 17 launches a step and at most nine left
    # the gradient of a layer's input reads the weights that the layer's update overwrites: never together
    for s in sets:
        assert not ({"dot_cf_64x64x48", "dot_ch_64x48x64"} <= set(s) or {"dot_bm_64x48x8", "dot_bo_48x8x64"} <= set(s)), s


def _args(text, label):
    line = re.search(rf"^\s*launch {label} .*args:(.*)$", text, re.M).group(1)
    return {int(b) for b in re.findall(r"#(\d+)", line)}


@pytest.mark.parametrize("build", [_mlp, lambda d: W.encoder_train(d, 64, 32, 4, 64, 2, seed=3), lambda d: W.encoder_train(d, 50, 40, 5, 72, 2, seed=3)],
                         ids=["perceptron", "encoder", "encoder-odd"])
def test_members_share_no_memory_that_one_of_them_writes(build):
    """Temporaries of launches that run at the same time have slots of their own (written ones: those whose slot another
    member of the set names through another buffer, or names at all and writes)."""
    text = _plan(build)
    slot = {int(b): int(s) for b, s in re.findall(r"#(\d+) temp \S+ elems=\d+ slot=(\d+)", text)}
    sets = _sets(text)
    assert sets
    for s in sets:
        owner = {}
        for label in s:
            for b in _args(text, label):
                if b in slot:
                    assert owner.setdefault(slot[b], b) == b, (s, label, b)


def _memory(text, written):
    """Per launch of a plan, in its order: (label, step, memory it names, memory it writes, buffers it names, buffers it writes);
    memory is a home buffer or a temporary's slot.  Members of a shared launch have one step.  `written`: per kernel, which of its
    arguments are no `const`."""
    slot = {int(b): int(s) for b, s in re.findall(r"#(\d+) temp \S+ elems=\d+ slot=(\d+)", text)}
    out, step, left = [], -1, 0
    for line in text.splitlines():
        head = re.match(r"\s*shared\d+_(\d+)x, one launch", line)
        m = re.match(r"\s*launch (\S+) \[\w+\] kernel=(\w+) .*args:(.*)$", line)
        if head:
            step, left = step + 1, int(head.group(1))
        if not m:
            continue
        if left:
            left -= 1
        else:
            step += 1
        args = m.group(3).split()
        assert len(args) == len(written[m.group(2)]), line
        names = [re.search(r"#(\d+)", x) for x in args]
        place = [None if x is None else ("slot", slot[int(x.group(1))]) if int(x.group(1)) in slot else ("home", int(x.group(1))) for x in names]
        named = [None if x is None else int(x.group(1)) for x in names]
        out.append((m.group(1), step, {x for x in place if x}, {x for x, w in zip(place, written[m.group(2)]) if x and w},
                    {x for x in named if x is not None}, {x for x, w in zip(named, written[m.group(2)]) if x is not None and w}))
    return out


def _hazards(launches, any_of, writes):
    """Pairs of launches of which one writes what the other names."""
    return [(i, j) for j, y in enumerate(launches) for i, x in enumerate(launches[:j]) if x[writes] & y[any_of] or x[any_of] & y[writes]]


@pytest.mark.parametrize("build", [_mlp, lambda d: _mlp(d, 300, (200, 330, 129, 7)), lambda d: W.encoder_train(d, 64, 32, 4, 64, 2, seed=3),
                                   lambda d: W.encoder_train(d, 50, 40, 5, 72, 2, seed=3)], ids=["perceptron", "perceptron-products", "encoder", "encoder-odd"])
def test_members_name_no_memory_that_another_one_writes(build, tmp_path, monkeypatch):
    """What a launch writes is read from its kernel's parameters.  No member of a shared launch names memory (a home buffer, or a
    temporary's slot) that another one writes; and two launches that depend on one another when each runs by itself are
    in the same order when some share."""
    from test_library_cpu import _compile_check
    monkeypatch.setenv("ADHIP_DUMP_CODE_DIR", str(tmp_path))
    monkeypatch.setenv("ADHIP_SHARE_INDEPENDENT", "0")
    proc, deps = build(OracleDevice()).finish()
    rc, msg = _compile_check(proc, deps)
    assert rc == 0, msg
    written = {}
    for p in tmp_path.glob("*.hip"):
        params = re.search(rf"__global__ [^{{;]*void {p.stem}\(const int\* __restrict__ guard,?([^{{]*)\) {{", p.read_text()) or \
            re.search(rf"__global__ [^{{;]*void {p.stem}\(const int\* guard,?([^{{]*)\) {{", p.read_text())
        written[p.stem] = ["*" in x and "const" not in x for x in params.group(1).split(",")]
    apart = _memory(lower_describe(proc, deps), written)
    monkeypatch.delenv("ADHIP_SHARE_INDEPENDENT")
    text = lower_describe(proc, deps)
    shared = _memory(text, written)
    assert _sets(text) and sorted(x[0] for x in shared) == sorted(x[0] for x in apart) and len({x[0] for x in apart}) == len(apart)
    for i, j in _hazards(shared, 2, 3):
        assert shared[i][1] < shared[j][1], (shared[i], shared[j])
    step = {x[0]: x[1] for x in shared}
    depends = _hazards(apart, 4, 5)   # by buffers: slots are others
    assert len(depends) > len(apart)
    for i, j in depends:
        assert step[apart[i][0]] < step[apart[j][0]], (apart[i], apart[j])


@pytest.mark.parametrize("build", [W.readme_mlp, lambda d: W.mlp_train(d, 3, (5, 4, 4, 2), 2)], ids=["readme", "perceptron"])
def test_phases_of_one_launch_share_memory_as_launches_do(build, monkeypatch):
    """A temporary whose last phase is over is memory for the phases behind it."""
    monkeypatch.setenv("ADHIP_SHARE_INDEPENDENT", "0")
    slots = lambda: int(re.search(r"temp slots: (\d+)", _plan(build)).group(1))  # noqa: E731
    together, text = slots(), _plan(build)
    assert "[merged]" in text
    monkeypatch.setenv("ADHIP_MERGE_SMALL", "0")
    assert together <= slots(), text


def test_kernels_of_shared_launches_are_counted():
    text = _plan(_mlp)
    own, shared, parts = map(int, re.search(r"kernels: (\d+) and (\d+) that run several of them as one launch, never compiled by themselves: (\d+)", text).groups())
    assert 0 < shared <= len(re.findall(r"^\s*shared\w+, one launch", text, re.M)) and parts <= own


def test_large_launches_stay_apart():
    text = _plan(lambda d: W.mlp_train(d, 4096, (4096, 4096, 4096, 1024), 2))
    for s in _sets(text):
        assert not any(label.startswith("dot") for label in s), s


def test_switched_off(monkeypatch):
    monkeypatch.setenv("ADHIP_SHARE_INDEPENDENT", "0")
    assert not _sets(_plan(_mlp))


@pytest.mark.parametrize("chains", [2, 20])
def test_a_program_that_fits_the_static_scratch_area_still_fits(chains):
    """What shares a launch shares no memory: chains of two products, 2 MB between them, of which 20 at a time would be more
    than the area holds."""
    cmds, keep = [], set()
    for i in range(chains):
        k = 64 + 4 * i   # no two of one shape: those would be one grouped launch
        cmds += [IR.CreateMat(np.zeros(1000 * k, np.float32), [1000, k], f"x{i}"), IR.CreateMat(np.zeros(k * 512, np.float32), [k, 512], f"v{i}"),
                 IR.CreateMat(np.zeros(512 * (8 + i), np.float32), [512, 8 + i], f"w{i}"),
                 IR.DotProduct(a=f"x{i}", b=f"v{i}", res=f"h{i}"), IR.DotProduct(a=f"h{i}", b=f"w{i}", res=f"y{i}")]
        keep.add(f"y{i}")
    text = lower_describe(IR.IRProcedure("main", cmds + [IR.EX()]), keep)
    assert bool(_sets(text)) == (chains == 2), text


# ---- on the GPU


@pytest.mark.gpu
@pytest.mark.parametrize("build", [_mlp, lambda d: _mlp(d, 100, (70, 90, 65, 10), 4), lambda d: _mlp(d, 300, (200, 330, 129, 7), 4),
                                   lambda d: W.encoder_train(d, 64, 32, 4, 64, 4, seed=3), lambda d: W.encoder_train(d, 130, 80, 5, 200, 4, seed=4)],
                         ids=["perceptron", "perceptron-odd", "perceptron-products", "encoder", "encoder-products"])
def test_shared_launches_match_launches_apart(build, hip_device, monkeypatch):
    """The same kernels, so the same bits, at the first pass (launched one by one) and at replays."""
    print("[case] shared launches", flush=True)
    def values(share):
        monkeypatch.setenv("ADHIP_SHARE_INDEPENDENT", share)
        out = []
        for _ in range(3):
            wl = build(hip_device)
            out.append({k: np.asarray(v.data, dtype=np.float32) for k, v in wl.run().items()})
        return out
    apart, shared = values("0"), values("1")
    for a, s in zip(apart, shared):
        for k in a:
            assert np.array_equal(a[k].view(np.uint32), s[k].view(np.uint32)), k
