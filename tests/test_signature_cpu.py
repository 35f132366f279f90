"""The autotune cache's key: the same for the same workload, another one for another
device, scene, count or generation of the batched kernels, so that a shape
tuned for earlier kernels is tuned again instead of replayed."""
import hashlib
import json
from types import SimpleNamespace

import numpy as np

from luxcore_amd import batch as B


def test_signature_names_the_kernels(monkeypatch):
    dev = SimpleNamespace(name="card")
    args = ([10000, 50000], [4096, 8192], "layout2")
    key = B.signature(dev, *args)
    assert key == B.signature(SimpleNamespace(name="card"), *args) and " " not in key
    others = [B.signature(SimpleNamespace(name="other"), *args), B.signature(dev, [10000], *args[1:]),
              B.signature(dev, args[0], [4096], "layout2"), B.signature(dev, args[0], args[1])]
    # the key of caches that hold no generation
    h = hashlib.sha1(dev.name.encode() + json.dumps(args[0]).encode() + np.asarray(args[1], np.int64).tobytes() + b"layout2")
    others.append(h.hexdigest()[:16])
    monkeypatch.setattr(B, "KERNELS", B.KERNELS + 1)
    others.append(B.signature(dev, *args))
    assert key not in others and len(set(others)) == len(others)
