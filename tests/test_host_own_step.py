"""Who takes the Newton step apart (solver._splits_assembly): only a program that has put nothing of its own in
the place of the assembly, of the line search or of the Newton step."""
import importlib

import pytest

pytest.importorskip("torch")


def _modules():
    return importlib.import_module("cpfem_amd.solver"), importlib.import_module("cpfem_amd.models")


def test_the_frameworks_own_class_and_functions():
    S, M = _modules()
    assert S._splits_assembly(M.CrystalPlasticity.__new__(M.CrystalPlasticity))
    assert not S._splits_assembly(object())


@pytest.mark.parametrize("name", ["line_search", "linear_incremental_solver"])
def test_a_function_in_the_place_of_the_modules(name, monkeypatch):
    S, M = _modules()
    own = getattr(S, name)
    monkeypatch.setattr(S, name, lambda *a: own(*a))
    assert not S._splits_assembly(M.CrystalPlasticity.__new__(M.CrystalPlasticity))


def test_an_assembly_in_the_place_of_the_classes(monkeypatch):
    S, M = _modules()
    own = M.CrystalPlasticity.assemble
    problem = M.CrystalPlasticity.__new__(M.CrystalPlasticity)
    problem.assemble = lambda *a, **k: own(problem, *a, **k)
    assert not S._splits_assembly(problem)
    sub = type("Sub", (M.CrystalPlasticity,), {"assemble": lambda self, *a, **k: own(self, *a, **k)})
    assert not S._splits_assembly(sub.__new__(sub))
    monkeypatch.setattr(M.CrystalPlasticity, "assemble", lambda self, *a, **k: own(self, *a, **k))
    assert not S._splits_assembly(M.CrystalPlasticity.__new__(M.CrystalPlasticity))
