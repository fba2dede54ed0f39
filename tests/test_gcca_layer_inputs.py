"""The input side of GCC-A's layers is uploaded once per particle number and device: a strategy that
is used under another current device uploads it there, as the permanents' own uploads do."""
import numpy as np
import torch


def test_layer_inputs_follow_the_current_device(monkeypatch):
    from theboss_amd import _device as D
    from theboss_amd.simulation_strategies import GeneralizedCliffordsSimulationStrategy

    class Calculator:
        matrix = np.eye(4, dtype=np.complex128)
        uploads = []

        def layer_inputs(self, S, weights):
            self.uploads.append((int(S[0].sum()), D.device()))
            return self.uploads[-1]

        def compute_layer_pmfs(self, inputs, prefixes):
            assert inputs == (int(prefixes[0].sum()) + 1, D.device())
            return torch.full(prefixes.shape, 0.25, dtype=torch.float64)

    here = {"device": torch.device("cuda", 0)}
    monkeypatch.setattr(D, "device", lambda index=None: here["device"])
    calculator = Calculator()
    strategy = GeneralizedCliffordsSimulationStrategy(calculator, np.random.default_rng(0))
    strategy.simulate([1, 1, 0, 0], 5)
    assert calculator.uploads == [(1, here["device"]), (2, here["device"])]
    here["device"] = torch.device("cuda", 1)
    strategy._calculate_layers([(0, 0, 0, 0)])  # the state is kept; only the device changed
    strategy._calculate_layers([(1, 0, 0, 0), (0, 1, 0, 0)])
    strategy._calculate_layers([(0, 0, 0, 1)])
    assert calculator.uploads[2:] == [(1, here["device"]), (2, here["device"])]
