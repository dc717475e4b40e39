"""Base of the operators' autograd functions."""
from torch.autograd import Function


class NativeFunction(Function):
    """A ``torch.autograd.Function`` whose ``apply`` runs the node of ``csrc/binding.cpp`` (``native``, the same arguments
    and results without the interpreter in the backward pass).  ``forward`` and ``backward`` do the same through ``_C``: they
    are there for callers that call them, and a subclass that overrides one of them is run through them."""
    _direct = False

    def __init_subclass__(cls, **kwargs):
        super().__init_subclass__(**kwargs)
        own = vars(cls)
        cls._direct = 'native' in own or cls._direct and not any(
            name in own for name in ('forward', 'backward', 'setup_context', 'jvp', 'vmap'))

    @classmethod
    def apply(cls, *args, **kwargs):
        return cls.native(*args, **kwargs) if cls._direct else super().apply(*args, **kwargs)
