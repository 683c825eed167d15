"""Host side of the engines without a GPU: the library call is a stub."""
import weakref

import numpy as np
import torch


def test_sir_run_holds_its_slots_across_the_call(monkeypatch):
    """abm_sir_run_watched launches steps for as long as it waits, and other
    threads allocate meanwhile: its count slots must not be free by then."""
    from jaxabm_amd.programs import sir

    slots_of, held = [], []

    class Lib:
        def abm_sir_run_watched(self, *args):
            held.append(slots_of[0]() is not None)
            return 0

    class Engine(sir.SIRNetworkEngine):
        def __init__(self):
            self.device, self.mode, self.t = torch.device("cpu"), 1, 0
            self.beta = self.gamma = 0.5
            self.rng = np.zeros(2, np.uint32)
            self._g = sir.SirGraph()
            self.state = self.mark = self.bitmaps = torch.zeros(1)
            self._watch = torch.zeros(2, dtype=torch.int32)
            self._stage = type("Stage", (), {"upload": staticmethod(torch.from_numpy)})

        def slot_buffer(self, steps):
            slots = torch.empty(steps)
            slots_of.append(weakref.ref(slots))
            return slots

    monkeypatch.setattr(sir, "lib", lambda: Lib())
    monkeypatch.setattr(sir, "ptr", lambda t: t.data_ptr())
    monkeypatch.setattr(sir, "stream_handle", lambda stream=None: None)
    eng = Engine()
    monkeypatch.setattr(eng, "_host_keys", lambda steps: np.zeros((steps, 4), np.int32))
    assert eng.run(3).shape == (3, 3)
    assert held == [True]
