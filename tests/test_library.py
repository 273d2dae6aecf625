"""The number by which the package refuses a kernel library that does not belong to it goes up with everything that the two
share. Host code only: no GPU needed."""
import hashlib

from lmsf_amd.ops import dispatch, library, program
from lmsf_amd.ops.hip_ops import HipOps

# One line a version, the newest last. A difference here means that an entry point, a structure, a route or a flag has
# changed: raise the number in csrc/runtime.hip and ops/library.py, then add its line (never change an old one).
VERSIONS = {38: "b3ef8bfa13f50e4e", 39: "a6516c9b237f5bb9", 40: "deeb2b301a468cfb",
            41: "6cebad8e9d1a97df", 42: "e35e1bf0818d5850", 43: "49e3e76bff5aa5a3"}


def shared() -> str:
    h = hashlib.sha256()
    for module in (library, program):
        for name, (res, args) in sorted(module._SIGNATURES.items()):
            h.update(repr((name, getattr(res, "__name__", None), [a.__name__ for a in args])).encode())
    for s in (dispatch.Tunables, dispatch.Route, dispatch.ProductShape, program.OpDesc, program.PlanInfo, program.StepDesc,
              program.TensorRef, program.CallbackArgs):
        h.update(repr((s.__name__, [(n, t.__name__) for n, t in s._fields_])).encode())
    routes = sorted((v, n) for n, v in vars(dispatch).items() if n.isupper() and isinstance(v, int))
    h.update(repr((routes, program.StepProgram.STAT_NAMES, HipOps.ATTENTION_WEIGHTS_F32, HipOps.ATTENTION_KEEP_PARTS)).encode())
    return h.hexdigest()[:16]


def test_the_version_follows_what_is_shared():
    assert (library.ABI_VERSION, shared()) == max(VERSIONS.items())
    assert library.load_library().lmsf_abi_version() == library.ABI_VERSION
