"""The host rules of the launches whose blocks wait for each other (csrc/resident_rules.hpp), compiled
for the host: what they must guarantee the kernels for every input."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RULES = os.path.join(REPO, "hr-weno_amd", "csrc", "resident_rules.hpp")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    """expr -> the value of a C++ expression over the rules, one compilation per program."""
    d = tmp_path_factory.mktemp("rules")

    def run(body):
        src, exe = d / "rules.cpp", d / "rules"
        src.write_text(f'#include <cstdio>\n#include "{RULES}"\nusing namespace hrw;\nint main()\n{{\n{body}\nreturn 0;\n}}\n')
        subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-o", str(exe), str(src)], check=True)
        out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
        return [[int(x) for x in line.split()] for line in out.splitlines()]
    return run


def test_one_step_in_place_needs_a_wait(rules):
    """Several blocks without maxima first wait for each other in the second step."""
    out = rules("for (int b = 0; b < 2; ++b) for (int a = 0; a < 2; ++a) for (int n = 1; n < 4; ++n)"
                ' std::printf("%d %d %d %d\\n", b, a, n, (int)resident_in_place(b, a, n));')
    for several, amax, n, ok in out:
        assert ok == (not several or amax or n > 1)


@pytest.mark.parametrize("most", [3, 64, 1024])
def test_launches_of_a_call(rules, most):
    """They add up to the call, none is longer than `most`, and none is a single step but in a call of one."""
    out = rules(f"for (int64_t n = 1; n < 5 * {most}; ++n) {{ for (int64_t l = n; l > 0;) {{ const int64_t s = launch_steps(l, {most});"
                ' std::printf("%lld ", (long long)s); l -= s; } std::printf("\\n"); }')
    for n, steps in enumerate(out, 1):
        assert sum(steps) == n and max(steps) <= most
        assert n == 1 or min(steps) >= 2


def test_blocks_of_a_batch_line_fit_the_device(rules):
    """One per CU at most, on whole devices and on partitions of them."""
    out = rules('for (int c = 1; c <= 512; ++c) std::printf("%d %d\\n", c, batch_line_blocks(c));')
    for cus, blocks in out:
        assert 1 <= blocks <= min(cus, 64) and (cus < 64 or blocks == 64)


def test_polls_from_the_environment(rules):
    """Whole decimal digits count; anything else leaves the usual number."""
    texts = {"0": 0, "1": 1, "300": 300, "2147483647": 2147483647, "": 77, "x": 77, "12x": 77, "-1": 77, " 3": 77,
             "2147483648": 77, "99999999999999999999": 77, "1e3": 77}
    body = "".join(f'std::printf("%d\\n", resident_polls("{t}", 77));' for t in texts)
    out = rules(body + ' std::printf("%d\\n", resident_polls(nullptr, 77));')
    assert [x[0] for x in out] == list(texts.values()) + [77]


def test_back_off(rules):
    """Calls that would wait in vain every time: few tries; one that does not, and the next is tried again."""
    out = rules("""
    BackOff b;
    int tries = 0;
    for (int call = 1; call <= 5000; ++call) {
        if (!b.skip()) {
            b.in_vain();
            ++tries;
            std::printf("%d\\n", call);
        }
    }
    int wait = 0;
    while (b.skip()) ++wait;
    b.went();
    std::printf("%d %d\\n", wait, (int)b.skip());
    b.in_vain();
    const int one = b.skip(), two = b.skip();
    std::printf("%d %d\\n", one, two);""")
    tries = [x[0] for x in out[:-2]]
    assert tries[:4] == [1, 3, 6, 11] and len(tries) < 30 and max(b - a for a, b in zip(tries, tries[1:])) == 257
    assert out[-2][0] <= 256 and out[-2][1] == 0 and out[-1] == [1, 0]


@pytest.mark.parametrize("first", [4, 0xffffffff - 300])
def test_exchange_numbers_leave_no_gap(rules, first):
    """Launches that are refused, wait in vain or go through, in any order: a maximum's word (one of
    four in turn, with bit 2 of the number) never reads as arrived before it is published."""
    out = rules(f"""
    ExchangeNumbers x;
    x.cleared();
    x.next = {first}u;
    unsigned word[4];
    // (as if all numbers before had been published)
    for (unsigned i = 1; i <= 4; ++i) word[(x.next - i) & 3] = x.next == kResFirstTag ? 0 : ((x.next - i) >> 2) & 1;
    unsigned long long seed = 1;
    for (int launch = 0; launch < 4000; ++launch) {{
        seed = seed * 6364136223846793005ull + 1442695040888963407ull;
        const unsigned used = 2 + (unsigned)(seed >> 33) % 13, what = (unsigned)(seed >> 50) % 4;
        if (x.need_clear(used)) {{
            for (unsigned &w : word) w = 0;
            x.cleared();
        }}
        if (what == 0) continue;              // refused: nothing is published
        for (unsigned q = 0; q < used; ++q) {{
            const unsigned tag = x.next + q, bit = (tag >> 2) & 1;
            if (word[tag & 3] == bit) std::printf("%d %u\\n", launch, tag);
            word[tag & 3] = bit;
        }}
        x.launched(used);
        if (what == 1) {{                      // some waited in vain: the words hold anything
            for (unsigned &w : word) w = (seed >> 40) & 1;
            x.lost();
        }}
    }}""")
    assert out == []
