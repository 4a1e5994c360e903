"""A minimal `Configurable` in the shape the kernel classes need.

AXLearn kernel classes are built as `cls.default_config().set(**kwargs).instantiate()`
(axlearn/common/flash_attention/utils.py:154). This module supplies just that protocol; it is not a
re-implementation of axlearn/common/config.py.
"""

from __future__ import annotations

import copy
import dataclasses
from typing import Any, Optional


def config_class(cls):
    """Marks a nested `Config` class; fields become dataclass fields."""
    return dataclasses.dataclass(cls)


# Values a shallow copy may share.  (A config is copied for every kernel instance of every call, and
# `copy.deepcopy` of its handful of plain fields took 15 us.)
_IMMUTABLE = frozenset((type(None), bool, int, float, str))


def _copy_config(cfg):
    """What `copy.deepcopy(cfg)` gives: a config that shares nothing mutable with `cfg`."""
    new = object.__new__(type(cfg))
    fields = new.__dict__
    fields.update(cfg.__dict__)
    for name, value in fields.items():
        if type(value) not in _IMMUTABLE and not isinstance(value, type):
            fields[name] = copy.deepcopy(value)
    return new


class Configurable:
    @config_class
    class Config:
        klass: Optional[type] = None

        def set(self, **kwargs) -> "Configurable.Config":
            for name in kwargs:
                if name not in self.__dataclass_fields__:
                    raise AttributeError(f"{type(self).__qualname__} has no field {name!r}")
            self.__dict__.update(kwargs)
            return self

        def clone(self, **kwargs) -> "Configurable.Config":
            return _copy_config(self).set(**kwargs)

        def instantiate(self, **kwargs) -> Any:
            return self.klass(self, **kwargs)

    @classmethod
    def default_config(cls) -> "Configurable.Config":
        return cls.Config(klass=cls)

    def __init__(self, cfg: "Configurable.Config"):
        self._config = _copy_config(cfg)

    @property
    def config(self) -> "Configurable.Config":
        return _copy_config(self._config)
