"""A loop that was shut down leaves no thread that still holds its engine."""

import weakref

from opsagent_amd.engine.engine import LLMEngine
from opsagent_amd.engine.serving import EngineLoop

from test_serving import CFG


def test_shutdown_ends_both_threads():
    loop = EngineLoop(LLMEngine(dict(CFG)))
    threads = (loop._thread, loop._watchdog)
    engine = weakref.ref(loop.engine)
    loop.shutdown()
    assert not any(t.is_alive() for t in threads)
    del loop
    import gc

    gc.collect()
    assert engine() is None       # gone on this thread, not whenever the watchdog wakes
