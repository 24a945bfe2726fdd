"""StepPlan.match (hostpath.cpp): which steps the native path takes, on CPU tensors.

match() may say yes only when the Python path would step exactly the batch's tensors with
these gradients: everything else is its refusal, after which the Python path rebuilds the
batch or raises.  No entry point of the library is called: the plans have none, or the test's.
"""
import ctypes
import subprocess
import threading
import time

import pytest
import torch

from morph_amd import _lib

SHAPES = [(4, 6), (5,), (0,), (3, 3)]


class Case:
    """Four parameters in two groups, a batch over all but the second."""

    def __init__(self, dtype=torch.float32, exports=False):
        self.params = [torch.nn.Parameter(torch.zeros(s)) for s in SHAPES]
        self.groups = [dict(params=self.params[:2], lr=1.0), dict(params=self.params[2:], lr=2.0)]
        self.present = [0, 2, 3]
        self.state = {p: dict(step=0, exp_avg=torch.zeros_like(p.data), exp_avg_sq=torch.zeros_like(p.data))
                      for p in self.params}
        self.dtype = dtype
        self.exports = [torch.zeros(s, dtype=torch.float16) for s in SHAPES] if exports else []
        self.array = (_lib.AdamwTensor * 3)()
        for d, i in zip(self.array, self.present):
            p = self.params[i]
            d.numel, d.param = p.numel(), p.data_ptr()
            d.exp_avg, d.exp_avg_sq = (self.state[p][k].data_ptr() for k in ("exp_avg", "exp_avg_sq"))
            d.out = self.exports[i].data_ptr() if exports else None
        self.plan = self.make_plan()

    def make_plan(self, entries=(0,) * 5):
        return _lib.hostpath().StepPlan(self.params, self.present, _lib.ctypes.addressof(self.array),
                                        _lib.dtype_code(self.dtype), -1, 0, 0, 0, list(entries))

    def grads(self):
        return [torch.ones(s, dtype=self.dtype) if i in self.present else None
                for i, s in enumerate(SHAPES)]

    def match(self, grads=None):
        before = [d.grad for d in self.array]
        ok = self.plan.match(self.groups, grads, self.exports, self.state)
        if not ok:
            assert [d.grad for d in self.array] == before  # a refusal writes nothing
        return ok


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind", [list, tuple])
def test_matching_gradients_are_taken_by_address(dtype, kind):
    c = Case(dtype, exports=True)
    for _ in range(2):
        gs = c.grads()
        assert c.match(kind(gs))
        assert [d.grad or 0 for d in c.array] == [gs[i].data_ptr() for i in c.present]
    address = gs[0].data_ptr()
    del gs  # the plan holds them until the next match or release()
    assert torch.ones(4, 6, dtype=dtype).data_ptr() != address
    c.plan.release()


def test_the_parameters_own_gradients():
    c = Case()
    for i in c.present:
        c.params[i].grad = torch.ones_like(c.params[i])
    assert c.match()
    assert c.array[0].grad == c.params[0].grad.data_ptr()
    c.params[1].grad = torch.ones(5)
    assert not c.match()  # a gradient more
    c.params[1].grad = None
    assert c.match()
    c.params[3].grad = None
    assert not c.match()  # one less


@pytest.mark.parametrize("change", [
    lambda c, g: g.__setitem__(0, None), lambda c, g: g.__setitem__(1, torch.ones(5)),
    lambda c, g: g.__setitem__(0, g[0].half()), lambda c, g: g.__setitem__(0, torch.ones(6, 4).t()),
    lambda c, g: g.__setitem__(0, torch.ones(4, 12)[:, ::2]), lambda c, g: g.__setitem__(3, torch.ones(8)),
    lambda c, g: g.__setitem__(3, torch.ones(10)), lambda c, g: g.__setitem__(3, g[3].to("meta")),
    lambda c, g: g.__setitem__(3, g[3].to_sparse()), lambda c, g: g.__setitem__(3, 1.0),
    lambda c, g: g.__setitem__(3, g[3].expand(1, 3, 3).expand(2, 3, 3)[:, 0]),
    lambda c, g: g.__setitem__(3, torch.ones(3, 3).as_subclass(type("Sub", (torch.Tensor,), {}))),
    lambda c, g: g.append(None), lambda c, g: g.pop(),
    lambda c, g: c.groups.reverse(), lambda c, g: c.groups.pop(),
    lambda c, g: c.groups[0]["params"].append(torch.nn.Parameter(torch.zeros(2))),
    lambda c, g: c.groups[1].__setitem__("params", [torch.nn.Parameter(p.data) for p in c.params[2:]]),
    lambda c, g: c.groups[1].__setitem__("params", tuple(c.params[2:])),
    lambda c, g: c.exports.__setitem__(3, torch.zeros(3, 3, dtype=torch.float16)),
    lambda c, g: c.exports.clear(), lambda c, g: c.exports.pop(),
    # a parameter that lies elsewhere, or is another size or layout where it lay
    lambda c, g: setattr(c.params[0], "data", torch.zeros(4, 6)),
    lambda c, g: setattr(c.params[3], "data", c.params[3].data[:2]),
    lambda c, g: setattr(c.params[3], "data", c.params[3].data.t()),
    # a moment replaced, moved, or gone
    lambda c, g: c.state[c.params[0]].__setitem__("exp_avg", torch.zeros(4, 6)),
    lambda c, g: c.state[c.params[3]].__setitem__("exp_avg_sq", torch.zeros(3, 3)),
    lambda c, g: setattr(c.state[c.params[3]]["exp_avg"], "data", torch.zeros(3, 3)),
    lambda c, g: c.state[c.params[3]].pop("exp_avg_sq"),
    lambda c, g: c.state.__setitem__(c.params[0], {k: v for k, v in c.state[c.params[3]].items()}),
    lambda c, g: c.state.pop(c.params[0]),
    lambda c, g: setattr(c, "state", {p: c.state[p] for p in reversed(c.params)}),
    lambda c, g: setattr(c, "state", None),
], ids=range(33))
def test_anything_else_is_refused(change):
    c = Case(exports=True)
    gs = c.grads()
    assert c.match(gs)
    change(c, gs)
    assert not c.match(gs)


def test_empty_views_of_a_larger_buffer_match():
    c = Case()
    empty = c.params[2]
    empty.data = torch.zeros(9)[4:4]
    c.state[empty] = dict(step=0, exp_avg=torch.zeros(8)[3:3], exp_avg_sq=torch.zeros(8)[8:])
    assert c.match(c.grads())


def test_other_containers_are_refused():
    c = Case()
    gs = c.grads()
    assert not c.match(iter(gs)) and not c.match(dict(enumerate(gs)))
    assert not c.plan.match(tuple(dict(g, params=iter(g["params"])) for g in c.groups), gs, [],
                            c.state)
    assert c.match(gs)


def test_other_views_with_the_same_layout_match():
    """A contiguous gradient of the right size is taken whatever its shape or offset, as in the
    Python path."""
    c = Case()
    gs = c.grads()
    gs[0] = torch.ones(24)
    gs[3] = torch.ones(10)[1:]
    assert c.match(gs) and c.array[2].grad == gs[3].data_ptr()


class Sub(torch.nn.Parameter):
    pass


def test_a_plan_over_subclass_parameters_refuses_their_own_gradients():
    """Parameters of a tensor subclass step on the Python path: no plan error on the way."""
    c = Case()
    sub = torch.zeros(4, 6).as_subclass(Sub)
    c.state = {sub if p is c.params[0] else p: s for p, s in c.state.items()}
    c.params[0] = c.groups[0]["params"][0] = sub
    c.array[0].param = sub.data_ptr()
    c.plan = c.make_plan()
    for i in c.present:
        c.params[i].grad = torch.ones(SHAPES[i])
    assert not c.match()


def test_a_plan_made_under_a_dispatch_mode_waits_for_its_end():
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    c = Case()
    gs = c.grads()
    with Mode():
        c.plan = c.make_plan()
        assert not c.match(gs)
    assert c.match(gs)


def test_launches_release_the_gil(tmp_path):
    """Other Python threads run while a launch waits (for room in a full queue, say): the entry
    points here wait, two seconds at most, for a word that another thread writes."""
    src = tmp_path / "entries.c"
    src.write_text("""
        #include <time.h>
        volatile int started, seen;
        int entry(void) {
          const time_t end = time(0) + 2;
          started = 1;
          while (!seen && time(0) <= end) { const struct timespec t = {0, 1000000}; nanosleep(&t, 0); }
          return seen ? 0 : -1;
        }""")
    lib = tmp_path / "entries.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    entries = ctypes.CDLL(str(lib))
    c = Case()
    c.plan = c.make_plan([ctypes.cast(entries.entry, ctypes.c_void_p).value] * 5)
    assert c.match(c.grads())
    started, seen = (ctypes.c_int.in_dll(entries, n) for n in ("started", "seen"))

    def answer():
        while not started.value:
            time.sleep(1e-3)
        seen.value = 1

    thread = threading.Thread(target=answer, daemon=True)
    thread.start()
    assert c.plan.launch(0, 0, False, 0, 0, 0, 0, 0) == 0
    thread.join()


@pytest.mark.parametrize("detector,adamw,closed", [(-1, 0, False), (0, -1, True), (0, 0, True)])
def test_launch_says_whether_the_detector_went_out(detector, adamw, closed):
    """The detector's launch carries the previous step's close: a step whose AdamW launch fails
    behind it has closed that step."""
    made = [ctypes.CFUNCTYPE(ctypes.c_int)(lambda rc=rc: rc) for rc in (detector, adamw)]
    det, upd = (ctypes.cast(f, ctypes.c_void_p).value for f in made)
    c = Case()
    c.plan = c.make_plan([det, det, upd, det, upd])
    assert c.match(c.grads()) and not c.plan.closed()
    assert c.plan.launch(0, 0, False, 0, 0, 0, 0, 0) == (detector or adamw)
    assert c.plan.closed() == closed


def test_places_tell_tensors_apart():
    places = _lib.hostpath().places
    t = torch.zeros(4, 6)
    of = lambda *ts: places(list(ts))  # noqa: E731
    assert of(t, t) == of(t, t.view(24)) and of(t) == of(torch.nn.Parameter(t))
    others = [t[:2], t[1:], t.t(), torch.zeros(4, 6), t.view(-1)[::2], t[:0]]
    assert len({of(t)} | {of(x) for x in others}) == 1 + len(others)
    assert of(t, others[0]) != of(others[0], t) and of() == b""
    with pytest.raises(TypeError):
        of(t, None)


def test_bad_plans_raise():
    p = [torch.zeros(3)]
    make = lambda present, entries=5: _lib.hostpath().StepPlan(  # noqa: E731
        p, present, _lib.ctypes.addressof((_lib.AdamwTensor * 2)()), 0, -1, 0, 0, 0, [0] * entries)
    for bad in ([], [1], [0, 0], [-1]):
        with pytest.raises(ValueError):
            make(bad)
    with pytest.raises(ValueError):
        make([0], 4)
