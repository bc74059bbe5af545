"""What the compiler made of the kernels, read in the assembly it prints for them, and the host side of what
the kernels compute with (no GPU needed)."""
import concurrent.futures
import os
import re
import subprocess

import pytest

from fused_attention_amd import build

HIPCC = os.path.join(build.ROCM, "bin", "hipcc")

# (head_dim, blocks of 16 rows per wave, key groups): two and three ring slots, one and two key groups, one sub-tile at a time
# and two.  The registers that a kernel may have come from where the launcher takes them.
GROUP_KERNELS = [(16, 1, 1), (16, 1, 2), (32, 1, 1), (32, 1, 2), (32, 2, 1), (64, 1, 1), (128, 1, 1), (128, 1, 2)]
ELEMENTS = ["fp16", "bf16"]


@pytest.fixture(scope="module")
def group_kernels(tmp_path_factory):
    """{(element, head_dim, NQ, GK, mode): ([lines of the kernel's assembly], {what its metadata say})}, unmasked (mode 0) and
    causal (2)."""
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    where = tmp_path_factory.mktemp("asm")

    def compiled(element):
        space = "fa::bf16" if element == "bf16" else "fa"
        source = ['#include "%s"' % os.path.join(build.CSRC, "fused_attn_kernel.hpp")]
        source += ["template __global__ void %s::fwd_kernel_group<%d, %d, %d, fa::%s, fa::group_waves_per_simd<%d, %d, false>()>(const fa::SplitParams);"
                   % (space, h, nq, gk, mode, h, nq) for h, nq, gk in GROUP_KERNELS for mode in ("kPlain", "kCausal")]
        (where / (element + ".hip")).write_text("\n".join(source) + "\n")
        subprocess.run([HIPCC] + build.HIPCC_FLAGS + ["--cuda-device-only", "-S", str(where / (element + ".hip")), "-o", str(where / (element + ".s"))],
                       check=True, capture_output=True)
        return (where / (element + ".s")).read_text()

    with concurrent.futures.ThreadPoolExecutor() as pool:
        texts = dict(zip(ELEMENTS, pool.map(compiled, ELEMENTS)))
    kernels = {}
    name = r"_ZN2fa(?:4bf16)?16fwd_kernel_groupILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E"
    for element, text in texts.items():
        lines = None
        for line in text.splitlines():
            found = re.match(name + r"\w+:", line)
            if found:
                lines = []
                kernels[(element,) + tuple(int(n) for n in found.groups())] = lines, {}
            elif line.startswith(".Lfunc_end"):
                lines = None
            elif lines is not None:
                lines.append(line.strip())
        for entry in text[text.index("amdhsa.kernels:"):].split("  - .agpr_count:")[1:]:
            found = re.search(r"\.name: +" + name, entry)
            kernels[(element,) + tuple(int(n) for n in found.groups())][1].update(
                (key, int(n)) for key, n in re.findall(r"\.(private_segment_fixed_size|vgpr_spill_count|vgpr_count): +(\d+)", entry))
    return kernels


def _loop_lines(lines):
    """The instructions of the blocks that the compiler marks as part of a loop, without those written by hand."""
    in_loop = by_hand = False
    for line in lines:
        if re.match(r"(\.LBB\d+_\d+:|; %bb\.)", line):
            in_loop = False
        in_loop = in_loop or (line.startswith((";", ".LBB")) and "Loop" in line)
        by_hand = "#ASMSTART" in line or (by_hand and "#ASMEND" not in line)
        if in_loop and not by_hand and line[:1] not in (";", ".", ""):
            yield line


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("H,NQ,GK", GROUP_KERNELS)
@pytest.mark.parametrize("element", ELEMENTS)
def test_the_group_kernel_waits_for_its_queries_once(group_kernels, H, NQ, GK, mode, element):
    # The key tiles come by loads written in assembly, with exact waits of their own, so that the only loads the compiler
    # knows of are the queries'.  A wait of its making inside a loop would be one for the key tiles on their way, in every pass.
    lines, _ = group_kernels[element, H, NQ, GK, mode]
    assert any("s_barrier" in line for line in _loop_lines(lines))
    assert [line for line in _loop_lines(lines) if line.startswith("s_waitcnt") and "vmcnt" in line] == []


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("H,NQ,GK", GROUP_KERNELS)
@pytest.mark.parametrize("element", ELEMENTS)
def test_the_group_kernel_keeps_its_values_in_registers(group_kernels, H, NQ, GK, mode, element):
    # None of its values pass through memory, with as many waves per SIMD as the launcher compiles it for (64 registers with
    # eight, 80 with six, 128 with four).
    _, said = group_kernels[element, H, NQ, GK, mode]
    assert said["private_segment_fixed_size"] == said["vgpr_spill_count"] == 0
    assert said["vgpr_count"] <= (64 if NQ == 1 and H <= 32 else 80 if NQ == 1 and H <= 64 else 128)


def test_division_by_multiplication_is_exact(tmp_path):
    # fa::Divisor as the kernels use it (the high half of n * mul, shifted), at every d up to 70, at every power of
    # two and its neighbours, and at the largest one: n on both sides of multiples of d, over the whole range.
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    (tmp_path / "div.hip").write_text('#include "%s"\n' % os.path.join(build.CSRC, "fused_attn_kernel.hpp") + r"""
#include <cstdio>
int main() {
    const int64_t most = 0x7fffffff;
    auto check = [&](int64_t d) {
        const fa::Divisor by = fa::divisor(d);
        auto right = [&](int64_t n) {
            const int64_t got = by.mul == 0 ? n : (int64_t)((((uint64_t)n * by.mul) >> 32) >> by.shift);
            if (got != n / d) std::printf("%lld / %lld is not %lld\n", (long long)n, (long long)d, (long long)got);
            return got == n / d;
        };
        const int64_t whole = most / d, step = whole / 1000 + 1;
        for (int64_t i = 0; i <= whole; i += step)
            for (int64_t n = i * d - 1; n <= i * d + 1; ++n)
                if (n >= 0 && n <= most && !right(n)) return false;
        for (int64_t n = whole * d - 1; n <= most && n <= whole * d + 1; ++n)
            if (n >= 0 && !right(n)) return false;
        return right(0) && right(d - 1) && right(most - 1) && right(most);
    };
    for (int64_t d = 1; d <= 70; ++d)
        if (!check(d)) return 1;
    for (int s = 1; s <= 31; ++s)
        for (int64_t d = ((int64_t)1 << s) - 1; d <= ((int64_t)1 << s) + 1 && d <= most; ++d)
            if (!check(d)) return 1;
    return check(most) ? 0 : 1;
}
""")
    subprocess.run([HIPCC] + build.HIPCC_FLAGS + [str(tmp_path / "div.hip"), "-o", str(tmp_path / "div")], check=True, capture_output=True)
    ran = subprocess.run([str(tmp_path / "div")], capture_output=True, text=True)
    assert ran.returncode == 0, ran.stdout
