"""MI355X-native FP8 grouped-expert path for PithTrain.

Same Python operator surface as ``pithtrain.operators`` for the hot path (FP8 quantisation,
grouped / dense FP8 linears, token permute with dedup, SwiGLU / bias epilogues); every kernel is
hand-written HIP for gfx950 behind the C-ABI in ``include/pithtrain_hip.h``.
"""

import os as _os

import torch as _torch

from . import _lib  # noqa: F401

# The backward runs on the thread that asks for it.  By default autograd hands every backward to a
# worker thread per device and waits for it; with one process per GPU that thread has nothing to run
# beside, and waking it and being woken by it cost 70-80 us a backward on the EPYC hosts of the
# MI355X (toy expert layer: 256 -> 172 us a step; 1001-token k/v linear: 171 -> 101 us).  The setting
# belongs to the importing thread; PITHTRAIN_AUTOGRAD_THREADS=1, or a later
# torch.autograd.set_multithreading_enabled(True), gives the worker threads back.
if _os.environ.get("PITHTRAIN_AUTOGRAD_THREADS", "0") != "1":
    _torch.autograd.set_multithreading_enabled(False)

__version__ = "0.1.0"
