"""One definition of a type across the library's translation units: the same
name for two types, templates or not, is undefined behaviour where the linker
merges what the units emit for them."""
import glob
import os
import re

from conftest import ROOT


def shared_types(text):
    """Names of the types a unit defines outside its anonymous namespaces."""
    text = re.sub(r"^namespace \{$.*?^\}  // namespace$", "", text, flags=re.M | re.S)
    return set(re.findall(r"^(?:struct|class|union|enum(?: class)?) (\w+)[^;]*?\{", text, flags=re.M))


def test_types_of_one_name():
    assert shared_types("struct A {\n};\nnamespace {\n\nstruct B {\n};\n\n}  // namespace\nstruct C;\n") == {"A"}
    units = glob.glob(os.path.join(ROOT, "tensomite.cr_amd", "csrc", "*.hip"))
    assert len(units) > 4
    seen = {}
    for unit in sorted(units):
        with open(unit) as f:
            for name in shared_types(f.read()):
                assert name not in seen, f"{name} in {os.path.basename(unit)} and {seen[name]}"
                seen[name] = os.path.basename(unit)
