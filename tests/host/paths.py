"""What the library's host code does with a solver, seen on the CPU with the
runtime of fake_hip.cpp: which kernels run, on which stream, with which
buffers.  Run as a program with the runtime's library and a scenario's name
(tests/test_host_paths.py builds the one and runs the others)."""
import ctypes as C
import os
import re
import sys

import numpy as np

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))
FAKE = None
DOFS, DOFS2, TINT, TINT2 = 0x100000, 0x200000, 0x300000, 0x400000  # stand for device arrays: nothing reads them


def start(lib):
    """Loads the fake runtime, then the library, whose HIP calls resolve to it."""
    global FAKE
    FAKE = C.CDLL(lib, mode=C.RTLD_GLOBAL)
    FAKE.fake_log.restype = C.c_char_p
    FAKE.fake_live.restype = FAKE.fake_bytes.restype = FAKE.fake_size.restype = C.c_size_t
    FAKE.fake_size.argtypes = FAKE.fake_capturing.argtypes = [C.c_void_p]


class Launch:
    def __getitem__(self, i):
        return "launch" if i == 0 else self.name

    def __init__(self, line):
        self.kernel, self.args = line.split()[1], dict(a.split("=") for a in line.split()[2:])
        self.stream = int(self.args["stream"], 16)
        m = re.search(r"(k_[a-z0-9_]+?)(?=[IiPvfdx])", self.kernel)
        self.name = m.group(1) if m else self.kernel
        m = re.search(r"k_sparseI(.)Li(\d)ELi(\d+)ELb(\d)ELb(\d)E", self.kernel)
        if m:
            self.name = "sparse " + {"01": "local", "10": "neigh", "11": "fused"}[m.group(4) + m.group(5)]

    def addr(self, what):
        return int(self.args[what], 16)


def events():
    """The runtime calls noted since the last time, in order."""
    out = []
    for line in FAKE.fake_log().decode().splitlines():
        assert not line.startswith(("free of", "allocation that")), line
        out.append(Launch(line) if line.startswith("launch") else tuple(line.replace("stream=", "").split()))
    FAKE.fake_clear()
    return out


def launches():
    return [e for e in events() if isinstance(e, Launch)]


def names():
    return [e.name for e in launches()]


def mesh(n=(3, 4, 3), jitter=0.1, **kw):
    from edge_amd import mesh as M
    return M.box(n, jitter=jitter, seed=5, **kw)


class Solver:
    def __init__(self, m, order, runs, precision, kernel=0):
        from edge_amd import _lib
        from edge_amd import setups as S
        self.L, self.m = _lib.lib(), m
        h, mi = C.c_void_p(), m.mesh_in()
        mat = [np.ascontiguousarray(a, np.float64) for a in S.random_materials(m.n_el, seed=5)]
        self.rc = self.L.edge_el_create(C.byref(_lib.ElConfig(order, runs, precision, kernel)), C.byref(mi),
                                        *[a.ctypes.data for a in mat], C.byref(h))
        self.h = h

    def info(self):
        k, f = C.c_int32(), C.c_int32()
        assert self.L.edge_el_kernel_info(self.h, C.byref(k), C.byref(f)) == 0
        return k.value, f.value

    def local(self, dofs=DOFS, t_int=TINT, stream=None):
        return self.L.edge_el_local(self.h, 0, self.m.n_el, 1e-3, dofs, t_int, stream)

    def neigh(self, dofs=DOFS, t_int=TINT, stream=None):
        return self.L.edge_el_neigh(self.h, 0, self.m.n_el, t_int, dofs, stream)

    def step(self, n, dofs=DOFS, t_int=TINT, stream=None, graph=0):
        return self.L.edge_el_step(self.h, n, 1e-3, dofs, t_int, graph, stream)

    def variant(self, kernel, flags):
        return self.L.edge_el_set_variant(self.h, kernel, flags)

    def close(self):
        assert self.L.edge_el_destroy(self.h) == 0


def one_run_without_factors():
    """One run whose flux solvers are found not to have rank 3: the element-
    batched data (and its projections) does not exist, so neither the default
    nor a variant may run on it, and no launch gets a null buffer."""
    for precision, order in ((32, 5), (32, 2), (64, 4), (64, 5)):
        FAKE.fake_setup_flags(8)
        s = Solver(mesh(), order, 1, precision)
        FAKE.fake_setup_flags(0)
        assert s.rc == 0
        assert s.info()[0] == (1 if precision == 32 else 4)
        assert s.variant(5, 3) != 0 and s.variant(5, 1) != 0
        events()
        for rc in (s.local(), s.neigh(), s.step(1), s.step(3)):
            assert rc == 0
        for e in launches():
            assert e.name != "sparse local" and e.name != "sparse neigh" and e.name != "sparse fused", e.kernel
        s.close()
        assert FAKE.fake_live() == 0


def general_forms_of_a_face():
    """What only the flux solvers can express stays off the sparse kernels:
    frames that the set-up kernel finds not to be orthonormal, a free surface
    between two elements, and faces whose elements are not each other's
    neighbours though every projection has one receiver."""
    for form in ("frames", "surface", "swap"):
        for precision, order, runs in ((32, 4, 1), (32, 3, 8), (32, 4, 16), (64, 4, 1), (64, 3, 16)):
            m = mesh()
            if form == "frames":
                FAKE.fake_setup_flags(16)
            elif form == "swap":
                for a in (m.el_fa_el, m.f_id, m.v_id):
                    a[5, 1], a[90, 2] = a[90, 2], a[5, 1]
            else:
                m.fa_type[np.argwhere((m.fa_el >= 0).all(axis=1))[9, 0]] = 101
            s = Solver(m, order, runs, precision)
            FAKE.fake_setup_flags(0)
            assert s.rc == 0
            events()
            for rc in (s.local(), s.neigh(), s.step(1), s.step(3)):
                assert rc == 0
            assert not [n for n in names() if n.startswith("sparse")], (form, precision, runs)
            s.close()
            assert FAKE.fake_live() == 0


def streams_do_not_share_projections():
    """Solvers of several runs whose neighbour step reads tInt: a step waits
    for the one before it, whatever its stream; separate local steps and
    steps that the caller captures leave the handle's projections alone."""
    a, b = 0x51, 0x52
    for precision, order, runs in ((32, 5, 8), (64, 3, 8), (64, 4, 16)):
        s = Solver(mesh(), order, runs, precision)
        assert s.info() == (5, 1)
        events()
        done = None
        for n, stream, graph in ((2, a, 0), (1, b, 0), (3, b, 0), (3, a, 0), (3, b, 1), (1, a, 1), (2, None, 0)):
            assert s.step(n, DOFS, TINT, stream, graph) == 0
            ev = events()
            sparse = [i for i, e in enumerate(ev) if isinstance(e, Launch) or e[0] == "graph"]
            assert sparse
            if done is not None:
                waits = [i for i, e in enumerate(ev) if e == ("wait", done, hex(stream or 0)[2:])]
                assert waits and waits[0] < sparse[0]
            rec = [i for i, e in enumerate(ev) if e[0] == "record"]
            assert len(rec) == 1 and rec[0] > sparse[-1] and ev[rec[0]][2] == hex(stream or 0)[2:]
            done = ev[rec[0]][1]
        assert s.local(DOFS2, TINT2, a) == 0 and s.neigh(DOFS2, TINT2, a) == 0
        ev = events()
        assert [e.name for e in ev if isinstance(e, Launch)][0] == "sparse local" and len(ev) == 2
        assert ev[0].addr("proj") == 0 and not ev[1].name.startswith("sparse")
        FAKE.fake_capturing(b)
        assert s.step(3, DOFS2, TINT2, b) == 0
        ev = events()
        assert all(isinstance(e, Launch) and e.stream == b for e in ev) and len(ev) == 6
        assert all(e.addr("proj") == 0 for e in ev if e.name == "sparse local")
        assert not [e for e in ev if e.name in ("sparse neigh", "sparse fused")]
        for n in (1, 3):  # a graph of the solver's own is refused there, and the caller's left alone
            assert s.step(n, DOFS2, TINT2, b, 1) != 0 and events() == []
            FAKE.hipGetLastError()
        FAKE.fake_capturing(None)
        s.close()
        assert FAKE.fake_live() == 0


def no_room():
    """Each allocation of the set-up failing in turn: the constants, maps, fault
    marks and projections of the sparse kernels leave a solver on the general
    kernels, with nothing of them kept; any other is an error.  Without room
    for the second projection buffer a multi-step call goes launch by launch."""
    from edge_amd import fault as FL
    for precision, order, runs, general in ((32, 3, 8, 1), (32, 4, 1, 5), (32, 3, 16, 2), (64, 3, 16, 1), (64, 4, 1, 5)):
        m = mesh((4, 4, 4), jitter=0)
        assert len(FL.tag_plane(m, 2, 0.5)) > 0
        s = Solver(m, order, runs, precision)
        full, k, left = FAKE.fake_bytes(), 0, []
        assert s.rc == 0, s.L.edge_last_error()
        s.close()
        while True:
            FAKE.fake_fail_after(k)
            s = Solver(m, order, runs, precision)
            fired = FAKE.fake_fail_after(-1) < 0
            FAKE.hipGetLastError()
            if not fired:
                assert s.rc == 0
                s.close()
                break
            if s.rc == 0:
                left.append(FAKE.fake_bytes())
                events()
                assert s.local() == 0 and s.neigh() == 0
                assert not [n for n in names() if n.startswith("sparse")] and s.info()[0] == general
                s.close()
            assert FAKE.fake_live() == 0
            k += 1
        # phys, maps, marks; projections too where the solver has no others
        assert len(left) == (4 if general == 1 else 3) and len(set(left)) == 1 and left[0] < full, (left, full)
    for precision, order, runs in ((32, 3, 8), (32, 4, 1), (64, 3, 16)):
        s = Solver(mesh(), order, runs, precision)
        events()
        FAKE.fake_fail_after(0)
        assert s.step(3) == 0
        FAKE.fake_fail_after(-1)
        assert names() == 3 * ["sparse local", "sparse neigh"]
        FAKE.fake_capturing(0x77)  # a capture on another stream goes on
        assert s.step(2, stream=0x51) == 0
        FAKE.fake_capturing(None)
        assert names() == ["sparse local", "sparse fused", "sparse neigh"]
        s.close()
        assert FAKE.fake_live() == 0


def autotuner_times_what_steps_run():
    """A candidate of n repetitions is launched as edge_el_step(n) launches it."""
    for precision, order, runs in ((32, 4, 1), (64, 4, 1), (32, 3, 8), (64, 3, 16), (32, 3, 16), (64, 5, 1)):
        s = Solver(mesh(), order, runs, precision)
        events()
        n, kernels, flags = C.c_int32(16), (C.c_int32 * 16)(), (C.c_int32 * 16)()
        ms = (C.c_double * 16)()
        assert s.L.edge_el_autotune(s.h, 1e-3, 3, None, C.byref(n), kernels, flags, ms) == 0
        ev = [e for e in events() if isinstance(e, Launch) or e[0] == "record"]
        marks = [i for i, e in enumerate(ev) if e[0] == "record"]
        timed = [[e.name for e in ev[a + 1:b]] for a, b in zip(marks[::2], marks[1::2])]
        assert len(timed) == n.value
        for i in range(n.value):
            assert s.variant(kernels[i], flags[i]) == 0
            assert s.step(3) == 0
            assert timed[i] == names(), (precision, runs, kernels[i], flags[i])
        s.close()
        assert FAKE.fake_live() == 0


def graphs_of_repeated_calls():
    """Kernel 5 captures a multi-step sequence when a call repeats the one
    before it; calls whose step counts or arrays take turns are launched, and a
    graph that is held is replayed whenever its call comes."""
    def kinds(s, n, dofs=DOFS):
        assert s.step(n, dofs, TINT, 0x51, 1) == 0
        return [e[0] for e in events() if e[0] in ("begin", "graph", "launch")]

    for precision, order, runs in ((32, 4, 1), (64, 4, 1), (32, 3, 8)):
        s = Solver(mesh(), order, runs, precision)
        events()
        run = lambda n: ["launch"] * (n + 1)
        assert kinds(s, 2) == run(2) and kinds(s, 3) == run(3) and kinds(s, 2) == run(2)
        assert kinds(s, 3, DOFS2) == run(3) and kinds(s, 3) == run(3)
        assert kinds(s, 3) == ["begin"] + run(3) + ["graph"]
        assert kinds(s, 3) == ["graph"] and kinds(s, 2) == run(2) and kinds(s, 3) == ["graph"]
        assert kinds(s, 1) == ["begin", "launch", "launch", "graph"] and kinds(s, 1) == ["graph"]
        assert kinds(s, 2) == run(2) and kinds(s, 1) == ["graph"]
        s.close()
        assert FAKE.fake_live() == 0


def more_waves_than_memory():
    """A number of plane waves that fits no memory is an error code."""
    s = Solver(mesh(), 3, 16, 32)
    one = np.zeros(14)  # (nothing is read before the device memory exists)
    live = FAKE.fake_live()
    rc = s.L.edge_el_error_norms(s.h, DOFS, 0, 2**31 - 1, one.ctypes.data, 0.0, None, None, None, None)
    assert rc != 0 and FAKE.fake_live() == live
    s.close()


def projections_exist():
    """Every launch of the sparse kernels has its constants, maps and
    projections, and a buffer large enough for them."""
    for precision, order, runs in ((32, 5, 1), (32, 3, 8), (32, 4, 16), (64, 4, 1), (64, 3, 8), (64, 4, 16)):
        s = Solver(mesh(), order, runs, precision)
        assert s.rc == 0
        events()
        for rc in (s.step(1), s.step(2), s.step(5)):
            assert rc == 0
        ls = launches()
        nv = (3 * order * (order + 1) // 2 + 3) // 4
        need = 16 * nv * runs * precision // 8 * s.m.n_el
        for e in ls:
            assert e.name.startswith("sparse"), e.kernel
            for a in ("phys", "rot"):
                assert FAKE.fake_size(e.addr(a)) > 0
            for a, used in (("proj", e.name != "sparse neigh"), ("proj_in", e.name != "sparse local")):
                assert not used or FAKE.fake_size(e.addr(a)) >= need, (e.kernel, a)
            assert e.name != "sparse fused" or e.addr("proj") != e.addr("proj_in")
        assert [e.name.split()[1] for e in ls] == (["local", "neigh", "local", "fused", "neigh", "local"] +
                                                   4 * ["fused"] + ["neigh"])
        s.close()
        assert FAKE.fake_live() == 0


if __name__ == "__main__":
    start(sys.argv[1])
    globals()[sys.argv[2]]()
