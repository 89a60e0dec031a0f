"""Host-side cache for 0-dim scale buffers.

Upstream reads ``self.a.item()`` on every forward (``torch_int/nn/linear.py:40-41``,
``nn/bmm.py:15``), a blocking device-to-host copy per call.  The buffers stay
(state-dict compatibility); this mixin remembers the Python float and only
re-reads when the buffer object or its version counter changed.
"""
import torch


class ScalarCacheMixin:
    def _scalar(self, name):
        buf = self._buffers.get(name)  # skips nn.Module.__getattr__: this runs several times per kernel launch
        if buf is None:
            buf = getattr(self, name)
            if not torch.is_tensor(buf):
                return float(buf)
        cache = self.__dict__.get("_scalar_cache")
        if cache is None:
            cache = self.__dict__["_scalar_cache"] = {}
        hit = cache.get(name)
        if hit is not None and hit[0] is buf and hit[1] == buf._version:
            return hit[2]
        value = float(buf.item())
        cache[name] = (buf, buf._version, value)
        return value


def read_scalars(pairs):
    """Fill the caches behind ``_scalar`` for (module, name) pairs whose floating-point buffers have one dtype and lie on one
    device with a single copy to the host (one that synchronises, like each ``item()`` it stands for); what does not fit is
    left to ``_scalar``."""
    found = []
    for mod, name in pairs:
        buf = mod._buffers.get(name)
        if torch.is_tensor(buf) and buf.is_cuda and buf.is_floating_point() and buf.numel() == 1:
            hit = mod.__dict__.setdefault("_scalar_cache", {}).get(name)
            if ((hit is None or hit[0] is not buf or hit[1] != buf._version)
                    and (not found or (buf.device == found[0][2].device and buf.dtype is found[0][2].dtype))):
                found.append((mod, name, buf, buf._version))
    if len(found) > 1:
        for (mod, name, buf, version), value in zip(found, torch.cat([f[2].reshape(1) for f in found]).tolist()):
            mod._scalar_cache[name] = (buf, version, value)
