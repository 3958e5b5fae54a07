"""The kernel library's C interface: its version moves with its prototypes, and the bindings pass what they take."""
import ctypes
import hashlib
import os
import re

from reinfer_amd.csrc import build
from reinfer_amd.kernels import library

# the prototypes' digest that goes with the version: where this fails, the interface has changed and needs the next version
VERSION, DIGEST = 34, "8c522cd3c913a08c"


def prototypes():
    with open(os.path.join(build.HERE, "reinfer_hip.h")) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    return text, {name: [] if args.strip() in ("", "void") else [re.sub(r"\s+", " ", a).strip() for a in args.split(",")]
                  for name, args in re.findall(r"\b(ra_\w+)\s*\(([^)]*)\)\s*;", text)}


def test_the_version_moves_with_the_prototypes():
    text, protos = prototypes()
    digest = hashlib.sha256(repr(sorted(protos.items())).encode()).hexdigest()[:16]
    stated = int(re.search(r"#define RA_ABI_VERSION (\d+)", text).group(1))
    assert (stated, digest) == (VERSION, DIGEST)
    assert library.ABI_VERSION == stated


def test_the_bindings_pass_what_the_prototypes_take():
    protos = prototypes()[1]
    kinds = {ctypes.c_int: r"(unsigned )?int \w+", ctypes.c_long: r"long (long )?\w+", ctypes.c_float: r"float \w+"}
    for name, args in library._SIGNATURES.items():
        assert len(args) == len(protos[name]), name
        for got, want in zip(args, protos[name]):
            assert got not in kinds or re.fullmatch(kinds[got], want), (name, want)
