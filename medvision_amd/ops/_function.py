"""Base of the operators' autograd functions."""
import torch
from torch.autograd import Function

_tracing = torch._C._get_tracing_state     # None outside of torch.jit.trace


class NativeFunction(Function):
    """A ``torch.autograd.Function`` whose ``apply`` runs the node of ``csrc/binding.cpp`` (``native``, the same arguments
    and results without the interpreter in the backward pass).  ``forward`` and ``backward`` do the same through ``_C``: for
    callers that call them, for a subclass that overrides one of them, and for ``torch.jit.trace``, which records a Python
    function as one node but of the native one nothing except the allocation of its result."""
    _direct = False

    def __init_subclass__(cls, **kwargs):
        super().__init_subclass__(**kwargs)
        own = vars(cls)
        cls._direct = 'native' in own or cls._direct and not any(
            name in own for name in ('forward', 'backward', 'setup_context', 'jvp', 'vmap'))

    @classmethod
    def apply(cls, *args, **kwargs):
        if cls._direct and _tracing() is None:
            return cls.native(*args, **kwargs)
        return super().apply(*args, **kwargs)
