"""A native call that stands for several methods of an object is right only while these are the package's own: a subclass, an
instance or a test may have put others in their place, which then have to run."""
from __future__ import annotations


class OwnMethods:
    """The methods ``names`` of ``cls`` as the package defines them; to be made where the class is defined."""

    def __init__(self, cls: type, *names: str) -> None:
        self.names = names
        self._methods = tuple((name, getattr(cls, name)) for name in names)

    def of_class(self, cls: type) -> bool:
        """Whether objects of ``cls`` run these very methods unless they hold others themselves."""
        for name, method in self._methods:
            if getattr(cls, name) is not method:
                return False
        return True

    def of(self, obj) -> bool:
        """Whether ``obj`` runs these very methods."""
        held = obj.__dict__
        for name in self.names:
            if name in held:
                return False
        return self.of_class(type(obj))
