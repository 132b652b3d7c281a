"""bench.py says how its steps ran: a lone system's steps are launched by the host whatever the
graph mode, so its line and its lone legs claim no graph replay (no GPU)."""
import ast
import pathlib

SOURCE = pathlib.Path(__file__).resolve().parent.parent / "bench.py"
LONE_LEGS = {"run_gpu", "run_drift", "run_c3", "run_c1", "run_per_call", "run_thermostats", "run_dump"}


def test_lone_legs_set_no_graph_mode():
    tree = ast.parse(SOURCE.read_text())
    legs = {f.name: f for f in tree.body if isinstance(f, ast.FunctionDef) and f.name in LONE_LEGS}
    assert set(legs) == LONE_LEGS
    for name, f in legs.items():
        calls = [n.func.attr for n in ast.walk(f) if isinstance(n, ast.Call) and isinstance(n.func, ast.Attribute)]
        assert "set_graph_mode" not in calls, name


def test_the_headline_config_claims_no_graph_replay():
    keys = [k.value for n in ast.walk(ast.parse(SOURCE.read_text())) if isinstance(n, ast.Dict)
            for k in n.keys if isinstance(k, ast.Constant)]
    assert "graph_replay" not in keys and keys.count("stepping") == 2  # the headline's and the ensemble's
