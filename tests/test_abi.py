"""liblcr.so loads and exports every function include/lcr.h declares; host-only
behaviour of the C ABI.  CPU only: no call here touches a GPU."""
import ctypes as C
import os
import re

import numpy as np

from conftest import ROOT


def declared_functions():
    text = open(os.path.join(ROOT, "include", "lcr.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = set(re.findall(r"\b(lcr_[a-z0-9_]+)\s*\(", text))
    return sorted(names)


def test_header_declares_expected_surface():
    names = declared_functions()
    for n in ("lcr_icp_create", "lcr_icp_set_source", "lcr_icp_set_target", "lcr_icp_align",
              "lcr_icp_final_transform", "lcr_icp_has_converged", "lcr_icp_fitness",
              "lcr_normals", "lcr_icp_batch_align", "lcr_last_error"):
        assert n in names


def test_library_exports_every_declared_symbol():
    lib = C.CDLL(os.path.join(ROOT, "lowcost3dreconstruction_amd", "liblcr.so"))
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, missing


def test_python_binding_lists_every_symbol():
    import lowcost3dreconstruction_amd as m
    assert sorted(m.EXPORTS) == declared_functions()


def test_params_default_are_pcl_defaults():
    import lowcost3dreconstruction_amd as m
    p = m.default_params()
    assert p.max_iterations == 10
    assert p.transformation_epsilon == 0.0
    assert p.euclidean_fitness_epsilon == -np.finfo(np.float64).max
    assert p.max_corr_dist == np.sqrt(np.finfo(np.float64).max)
    assert p.point_to_plane == 0


def test_invalid_params_rejected_before_any_device_call():
    import lowcost3dreconstruction_amd as m
    p = m.default_params()
    p.max_iterations = 0  # fine_registration.cpp:76-78 rejects this
    h = C.c_void_p()
    rc = m.lib.lcr_icp_create(C.byref(p), C.byref(h))
    assert rc == -1
    assert b"greater than zero" in m.lib.lcr_last_error()


def header_struct_fields(name):
    """Field names, in order, of `typedef struct { ... } name;` in lcr.h."""
    text = open(os.path.join(ROOT, "include", "lcr.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    m = re.search(r"typedef struct\s*\{([^{}]*)\}\s*" + name + r"\s*;", text)
    assert m, name
    fields = []
    for decl in m.group(1).split(";"):
        decl = decl.strip()
        if decl:
            fields.append(re.findall(r"([A-Za-z_][A-Za-z0-9_]*)\s*(?:\[[^\]]*\])?\s*$", decl)[0])
    return fields


def test_python_structs_mirror_the_header():
    import lowcost3dreconstruction_amd as lcr
    for cname, py in (("lcr_icp_params", lcr.IcpParams), ("lcr_cycle_desc", lcr.CycleDesc),
                      ("lcr_cycle_result", lcr.CycleResult), ("lcr_tune_result", lcr.TuneResult)):
        assert [f for f, _ in py._fields_] == header_struct_fields(cname), cname


def test_cycle_wrapper_fills_every_descriptor_field():
    """Every lcr_cycle_desc field is set by Cycle.__init__ from a name it defines."""
    import inspect
    import lowcost3dreconstruction_amd as lcr
    src = inspect.getsource(lcr.Cycle.__init__)
    params = set(inspect.signature(lcr.Cycle.__init__).parameters)
    for f, _ in lcr.CycleDesc._fields_:
        assert re.search(r"\bd\." + f + r"\s*=", src), f
    for name in re.findall(r"int\(bool\((\w+)\)\)", src):
        assert name in params, name
    assert {"hyp_gate", "precision_mode", "proposal", "n_hyp", "guesses"} <= params


def test_bench_times_runs_after_the_capture(monkeypatch):
    """A handle's second run captures its graphs; what bench.py times comes after it."""
    import sys
    sys.path.insert(0, ROOT)
    import bench

    class Cycle:
        runs = 0

        def run(self):
            self.runs += 1

    c = Cycle()
    ticks = []
    monkeypatch.setattr(bench.time, "perf_counter", lambda: ticks.append(c.runs) or float(c.runs))
    assert bench.timed_steps(c, 3) == 1.0
    assert ticks == [2, 5]
