"""Matrix products that are written out in a kernel (inline assembly) are unknown to the compiler as such: it keeps none of the
distances that its own products get.  What the source arranges instead is looked at in the assembly, along every path."""
import re
import subprocess

import pytest

from palm_infra_amd.kernels import library

# v_mfma_f32_16x16x32_bf16 holds the matrix cores for four issue slots.  Its result may be read or written over by another instruction nine slots
# behind it (eight between them); the kernel keeps four products between.  Its operands are to be two slots old when they were
# written by a vector instruction.
PRODUCT, SLOTS, RESULT, OPERAND = "v_mfma_f32_16x16x32_bf16", 4, 1 + 4 * 4, 2


def assembly(source, defines, out):
    cmd = [library._hipcc(), *library.flags_of(source), *[f"-D{d}" for d in defines], "--cuda-device-only", "-S", str(library.CSRC / source), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True, text=True)
    return out.read_text()


def registers(operand):
    m = re.fullmatch(r"-?\|?([va])(?:(\d+)|\[(\d+):(\d+)\])\|?", operand.strip())
    if not m:
        return set()
    first, last = (int(m[2]), int(m[2])) if m[2] else (int(m[3]), int(m[4]))
    return {(m[1], i) for i in range(first, last + 1)}


class Instruction:
    def __init__(self, text, written_out):
        self.text = text
        self.name, _, rest = text.partition(" ")
        operands = [p.split()[0] if p.split() else "" for p in re.sub(r"\s+", " ", rest).split(",")]
        sets = [registers(o) for o in operands]
        writes_first = not re.match(r"(s_|v_cmp|ds_write|global_store|scratch_store|flat_store|buffer_store|global_load_lds)", self.name)
        self.writes = sets[0] if writes_first and sets else set()
        self.reads = set().union(*(sets[1:] if writes_first else sets)) if sets else set()
        self.product = self.name == PRODUCT
        self.written_out = written_out and self.product
        self.vector = self.name.startswith("v_") and not self.name.startswith("v_mfma")
        self.sum = sets[3] if self.product else set()                   # (a product's third source)
        self.target = rest.strip() if self.name.startswith(("s_cbranch", "s_branch")) else None
        self.sleeps = int(rest, 0) + 1 if self.name == "s_nop" else 1


def kernel(text, name):
    """The kernel's instructions and, for each, those that may come next."""
    lines = iter(text.splitlines())
    for line in lines:
        if re.match(rf"_Z\w*{name}\w*:", line):
            break
    else:
        raise AssertionError(f"no kernel {name}")
    code, labels, written_out = [], {}, False
    for line in lines:
        if line.startswith(".Lfunc_end"):
            break
        if "#ASMSTART" in line or "#ASMEND" in line:
            written_out = "#ASMSTART" in line
            continue
        line = line.split(";")[0].rstrip()
        label = re.match(r"(\.\w+):", line)
        if label:
            labels[label[1]] = len(code)
        elif line.startswith("\t") and not line.strip().startswith("."):
            code.append(Instruction(line.strip().replace("\t", " "), written_out))
    following = []
    for i, one in enumerate(code):
        after = [] if one.name in ("s_branch", "s_endpgm") else [i + 1]
        if one.target:
            after.append(labels[one.target])
        following.append([j for j in after if j < len(code)])
    return code, following


def too_near(code, following):
    """What reads or writes a written-out product's result with too little on purpose in between (products, s_nop; what happens to stand there
    does not count), and vector instructions that write its operands just before it."""
    found = []
    for i, one in enumerate(code):
        if one.written_out:
            seen, todo = {}, [(j, 1) for j in following[i]]
            while todo:
                j, slots = todo.pop()
                if slots >= RESULT or seen.get(j, RESULT) <= slots:
                    continue
                seen[j] = slots
                other = code[j]
                touched = (other.reads | other.writes) & one.writes
                if touched and not (other.product and not (other.reads - other.sum) & one.writes):
                    found.append(f"{other.text}   [{slots} behind {one.text}]")
                    continue
                more = SLOTS if other.product else other.sleeps if other.name == "s_nop" else 0
                todo += [(k, slots + more) for k in following[j]]
        elif one.vector and one.writes:
            todo = [(j, 0) for j in following[i]]
            while todo:
                j, slots = todo.pop()
                if slots >= OPERAND:
                    continue
                other = code[j]
                if other.written_out and other.reads & one.writes:
                    found.append(f"{other.text}   [operand by {one.text}]")
                todo += [(k, slots + other.sleeps) for k in following[j]]
    return found


@pytest.fixture(scope="module")
def large_tiles(tmp_path_factory):
    return {source: assembly(source, [], tmp_path_factory.mktemp("assembly") / f"{source}.s") for source in ("linear_big.hip", "moe_grouped.hip")}


@pytest.mark.parametrize("source,name,products", [("linear_big.hip", f"linear_big_kernelILi{nt}ELb{gated}E", 32 * nt) for nt in (2, 3, 4) for gated in (0, 1)]
                         + [("moe_grouped.hip", f"moe_big_kernelILi{nt}ELi{form}E{to}", 32 * nt) for nt in (1, 2, 3) for form, to in ((0, "f"), (0, "6bf16_t"), (2, ""))]
                         + [("moe_grouped.hip", f"moe_big_kernelILi4ELi{form}E{to}", 16 * (8 + 7 + 6 + 5 + 4))                # a walk for each number of columns
                            for form, to in ((0, "f"), (0, "6bf16_t"), (1, ""), (2, ""), (3, ""), (4, ""))])
def test_large_tiles_keep_their_products_distances_and_keep_nothing_in_memory(large_tiles, source, name, products):
    code, following = kernel(large_tiles[source], name)
    assert sum(one.written_out for one in code) == products
    assert too_near(code, following) == []
    assert not any(one.name.startswith("scratch_") for one in code)


@pytest.fixture(scope="module")
def attention_of_heads_of_128(tmp_path_factory):
    return assembly("attention_mfma.hip", ["PALM_HEAD_DIM=128"], tmp_path_factory.mktemp("assembly") / "attention.s")


@pytest.mark.parametrize("prescaled", [1, 0])
def test_wide_attention_keeps_its_products_distances(attention_of_heads_of_128, prescaled):
    code, following = kernel(attention_of_heads_of_128, f"attention_prefill_wide_kernelILb{prescaled}E")
    assert sum(one.written_out for one in code) == 4 * 34
    assert too_near(code, following) == []


@pytest.mark.parametrize("prescaled", [1, 0])
def test_wide_attention_waits_for_loads_where_it_says_so_and_keeps_nothing_in_memory(attention_of_heads_of_128, prescaled):
    """Between the first product and the last the loads into LDS, which the compiler does not know, stay on their way: all of them are waited
    for behind a read of the page table only, once in 64 pages."""
    name = f"attention_prefill_wide_kernelILb{prescaled}E"
    code, _ = kernel(attention_of_heads_of_128, name)
    assert not any(one.name.startswith("scratch_") for one in code)
    products = [i for i, one in enumerate(code) if one.written_out]
    waits = [i for i, one in enumerate(code) if one.name == "s_waitcnt" and "vmcnt" in one.text and products[0] < i < products[-1]]
    of_the_table = [i for i in waits if "vmcnt(0)" in code[i].text and code[i - 1].name == "global_load_dword"]
    assert len(of_the_table) <= 1 and ["vmcnt(8)" in code[i].text for i in waits if i not in of_the_table] == [True]
