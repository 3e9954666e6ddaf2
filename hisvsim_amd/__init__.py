"""hisvsim_amd -- MI355X-native hierarchical state-vector simulation.

The compute path is libhsv.so (HIP kernels for gfx950 behind the C ABI in
include/hsv.h). Two Python front ends sit on it:

* ``hisvsim_amd.svsimulator_py_wrapper`` -- the reference's pybind module API
  (StateVector, AggregateGate_*, BoundGate, gather_and_execute_on, ...);
* ``hisvsim_amd.capi`` -- a thin ctypes binding of the C ABI.

Build both in place with ``python -m hisvsim_amd.build``.
"""
import importlib
import importlib.machinery
import importlib.util
import os
import sys
import threading

HERE = os.path.dirname(os.path.abspath(__file__))
MODULE = "svsimulator_py_wrapper"
_load_lock = threading.Lock()


def own_module():
    """The in-tree pybind module for the package's own use, with sys.path left
    alone (the package's folder on it would hide a program's own modules of
    the same names): None if it is not built, or if another module of its name
    is loaded."""
    path = os.path.realpath(HERE)
    with _load_lock:
        if MODULE in sys.modules:
            file = getattr(sys.modules[MODULE], "__file__", None)
            return sys.modules[MODULE] if file and os.path.realpath(os.path.dirname(file)) == path else None
        spec = importlib.machinery.PathFinder.find_spec(MODULE, [HERE])
        if spec is None:
            return None
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        sys.modules[MODULE] = module
        return module


def load_module():
    """Imports the in-tree pybind module (raises ImportError if not built)."""
    if HERE not in sys.path:
        sys.path.insert(0, HERE)
    return importlib.import_module(MODULE)


__all__ = ["load_module"]
