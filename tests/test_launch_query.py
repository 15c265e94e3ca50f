"""Asking an engine whether a launch is possible sets nothing (no GPU)."""


def test_launch_query_sets_nothing(monkeypatch):
    from idmx import _lib
    from idmx.LBM._engine import SCEngine
    calls = []

    def call(name, *args):
        calls.append(name)
        if name == 'idmx_sc_launch_ok':
            args[-1]._obj.value = int(args[4] != 9)
    monkeypatch.setattr(_lib, 'call', call)
    eng = SCEngine.__new__(SCEngine)
    eng.handle = None
    assert eng.launch_ok(64, 4, 8, 1) is True and eng.launch_ok(256, 2, 8, 9) is False
    assert set(calls) == {'idmx_sc_launch_ok'}
