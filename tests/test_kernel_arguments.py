"""Interfaces that the kernel source and the host keep alike by hand: the structures that
say where a kernel's by-value modifications lie among its arguments, the number of them,
and the records that host and kernels share."""
import os
import re

import pytest

import sandengine_amd as S

CSRC = os.path.join(os.path.dirname(S.__file__), "csrc")


def source(name):
    with open(os.path.join(CSRC, name)) as f:
        return re.sub(r"//[^\n]*", "", f.read()).replace("\\\n", "\n")


def size_class(t):
    """What an argument of type t takes: a pointer, a whole number or a structure."""
    t = t.replace("const", "").replace("__restrict__", "").strip()
    return "pointer" if "*" in t else {"u32": "int", "int": "int", "u64": "long"}.get(t.split()[0], t.split()[0])


def fields(text, struct):
    body = re.search(r"struct %s \{(.*?)\n\};" % struct, text, re.S).group(1)
    out = []
    for decl in filter(None, (d.strip() for d in body.split(";"))):
        first, *rest = decl.split(",")
        base = re.match(r"((?:const )?\w+(?: char)?)\s*(.*)", first)
        for item in [base.group(2)] + rest:
            out.append(size_class(base.group(1) + ("*" if "*" in item else "")))
    return out


def parameters(text, kernel):
    args = re.search(kernel + r"\((.*?)\)\s*\{", text, re.S).group(1)
    return [size_class(a.strip()) for a in args.split(",")]


@pytest.mark.parametrize("file,kernel,struct", [
    ("se_kernels.hip", r"se_step_plain_r##R##_nt##NT", "se_plain_args"),
    ("se_kernels.hip", r"se_frame_b##B", "se_frame_args"),
    ("se_sliced.hip", r"se_sl_brush", "se_slbrush_args")])
def test_argument_structures_follow_the_parameters(file, kernel, struct):
    text = source(file)
    got = parameters(text, kernel)
    assert got[-1] == "se_few" and got == fields(text, struct)


def test_modifications_by_value():
    n = re.search(r"#define SE_PLAIN_MODS (\d+)", source("se_kernels.hip")).group(1)
    assert n == re.search(r"kFewMods = (\d+);", source("se_internal.hpp")).group(1)


@pytest.mark.parametrize("struct,host,file", [("se_slgrid", "SlicedGrid", "se_sliced.hpp"), ("se_slworld", "SlicedWorld", "se_sliced.hpp"),
                                              ("se_slknown", "SlicedKnown", "se_sliced.hpp"), ("se_fillspec", "FillSpec", "se_internal.hpp")])
def test_shared_records_have_the_same_fields(struct, host, file):
    kernel = source("se_kernels.hip" if struct == "se_fillspec" else "se_sliced.hip")

    def names(text, s):
        body = re.search(r"struct %s \{(.*?)\n\s*\};" % s, text, re.S).group(1)
        return [re.match(r"[\s*]*(\w+)", re.sub(r"^\s*(?:const )?(?:unsigned char|\w+)[\s*]+", "", item) if j == 0 else item).group(1)
                for decl in filter(None, (d.strip() for d in body.split(";"))) for j, item in enumerate(decl.split(","))]
    assert names(kernel, struct) == names(source(file), host)
