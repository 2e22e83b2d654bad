"""The host path (csrc/torch_ops.cpp) on the CPU, for tests of what it does with autograd, errors
and argument checks: the module is compiled from the same source with the device test and the
stream query exchanged, and every entry of the C ABI is the oracle's function of the same name."""
import importlib.util
import os
import re
import subprocess

import oracle
from custom_helper_op_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "chop_costvol.h")

_FILL = """  const int rc = {base}({args});
  const int64_t entries = B * H * W * D * {per_entry}, inner = {inner};
  for (int64_t i = 0; rc == 0 && i < entries; ++i)
    if (reduce == 0 ? mask[i] <= 0 : mask[i] < 0)
      for (int64_t j = 0; j < inner; ++j) cost[i * inner + j] = *default_cost;
  return rc;"""
_FILL_GRAD = """  *default_grad = 0;
  for (int64_t i = 0; i < mask_count * inner; ++i)
    if (reduce == 0 ? mask[i / inner] <= 0 : mask[i / inner] < 0) *default_grad += out_grad[i];
  return 0;"""


def _entry(kind, name, params):
    """One function of the C ABI as C++ source."""
    names = [re.search(r"(\w+)$", p).group(1) for p in params]
    at, before, types = dict(zip(names, params)), "", list(params)
    body = "  return (%s)CHOP_ERR_NO_DEVICE;" % kind
    of_oracle = name.replace("chop_", "chop_oracle_", 1)
    if "_fwd_fill_f" in name:
        v2 = "_v2_" in name
        body = _FILL.format(base=name.replace("_fill", ""),
                            args=", ".join(n for n in names if n != "default_cost"),
                            per_entry="(reduce == 0 ? 1 : groups)" if v2 else "1",
                            inner="(reduce == 0 ? groups : 1)" if v2 else "1")
    elif re.search(r"default_fill_grad_f\d\d$", name):
        body = _FILL_GRAD
    elif re.search(r"_(fwd|bwd)_f\d\d$", name):
        types = [t.replace("int groups", "int64_t groups") for t in types[1:]]
        before = "int %s(%s, int);\n" % (of_oracle, ", ".join(types))
        args, scratch = names[1:], ""
        for n in ("base_plane_grad", "depth_grid_grad"):  # may be null here, not in the oracle
            if n in at:
                real = "float" if "float" in at[n] else "double"
                scratch = "  std::vector<%s> unused(B * H * W * D);\n" % real
                args = ["(%s ? %s : unused.data())" % (n, n) if a == n else a for a in args]
        body = scratch + "  return %s(%s, 1);" % (of_oracle, ", ".join(args))
    return ("%s%s %s(%s) {\n  if (chop_test_status) return (%s)chop_test_status;\n%s\n}\n"
            % (before, kind, name, ", ".join(params), kind, body))


def c_abi_source():
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    out = ["#include <vector>\nextern \"C\" {\nint chop_test_status = 0;  // returned by every entry, if set\n"
           "const char *chop_last_error_string(void) { return \"as the test asked\"; }\n"]
    for kind, name, params in re.findall(r"^(int|size_t) (chop_\w+)\(([^)]*)\);", text, flags=re.M):
        params = [] if params == "void" else [" ".join(p.split()) for p in params.split(",")]
        out.append(_entry(kind, name, params))
    return "".join(out) + "}\n"


def host_source():
    text = open(os.path.join(build.CSRC, "torch_ops.cpp")).read()
    for there, here in (("#include <c10/hip/HIPStream.h>\n", ""),
                        ("../../include/chop_costvol.h", HEADER),
                        ("static_cast<void *>(c10::hip::getCurrentHIPStream(t.device().index()).stream())",
                         "(void)t, nullptr"),
                        ("if (!t.is_cuda())", "if (!t.is_cpu())")):
        assert text.count(there) == 1, there
        text = text.replace(there, here)
    return text + c_abi_source()


def build_module(folder):
    """Compiles the CPU form into `folder` and imports it."""
    oracle.build()
    source, so = (os.path.join(str(folder), n) for n in ("torch_ops_cpu.cpp", "_chop_torch.so"))
    with open(source, "w") as f:
        f.write(host_source())
    compile_, link = build.torch_module_commands()
    at = compile_.index("-c")
    flags = [x for x in compile_[1:at] if x not in ("-O2", "-Wall")]
    libs = [x for x in link[link.index("-o") + 2:] if x.startswith(("-L", "-lc10", "-ltorch")) and x != "-lc10_hip"]
    where = os.path.join(ROOT, "oracle")
    subprocess.run(["g++", "-O0", *flags, "-shared", source, "-o", so, *libs, "-L" + where, "-l:libchop_oracle.so",
                    "-Wl,-rpath," + where], check=True)
    spec = importlib.util.spec_from_file_location("_chop_torch", so)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module, so
