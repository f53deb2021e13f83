"""The delta form's kv runs as the kernels decode them: decode_fitted and decode_line of csrc/hstu_common.h, compiled for the host.  Needs no GPU.

A wave is run lane by lane: a lane stops at the first instruction across lanes whose other operands are not known yet; when all have, its result is
known and they start over."""

import os
import shutil
import subprocess

import pytest

_HARNESS = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include <tuple>
#include <vector>
#define __device__
#define __forceinline__
#define HSTU_CONST(T, p) ((const T*)(p))
struct { int x; } threadIdx;
struct DecodeParams {
    const void* offsets;
    int num_mb, B, H, max_seq_len, offsets_i64, delta, fit_runs, line_weight, line_wgs;
    unsigned mb_magic, mb_shift;  // the divisor itself: fast_div's constants have tests of their own on the device
};
struct Work {
    int b, h, split, nsplit, jt_begin, jt_end, fit_slot;
    bool operator==(const Work& o) const {
        return std::tie(b, h, split, nsplit, jt_begin, jt_end, fit_slot) == std::tie(o.b, o.h, o.split, o.nsplit, o.jt_begin, o.jt_end, o.fit_slot);
    }
};
int fast_div(int x, unsigned d, unsigned) { return x / (int)d; }
void fail(const char* what) { printf("%s\n", what), exit(1); }

struct Stop {};
std::vector<std::vector<int64_t>> known;  // operands of the instructions across lanes so far, by lane
std::vector<int64_t> pending(64);
size_t at;
const std::vector<int64_t>& across(int64_t v) {
    if (at < known.size()) return known[at++];
    pending[threadIdx.x] = v;
    throw Stop();
}
int wave_inclusive_scan(int v) {
    const auto& a = across(v);
    int64_t s = 0;
    for (int l = 0; l <= threadIdx.x; ++l) s += a[l];
    return (int)s;
}
int readlane(int v, int lane) { return (int)across(v)[lane]; }
uint64_t ballot(bool v) {
    const auto& a = across(v);
    uint64_t m = 0;
    for (int l = 0; l < 64; ++l) m |= (uint64_t)(a[l] != 0) << l;
    return m;
}
#define __builtin_amdgcn_readlane readlane
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __ballot ballot
#define __popcll __builtin_popcountll
SOURCE

template <class F>
bool wave(F decode, Work& w) {
    known.clear();
    while (true) {
        int ended = 0;
        bool got = false;
        for (threadIdx.x = 0; threadIdx.x < 64; ++threadIdx.x) {
            at = 0;
            Work mine{-1, -1, -1, -1, -1, -1, -1};
            try {
                const bool r = decode(mine);
                if (ended++ && (r != got || (r && !(mine == w)))) fail("lanes disagree");
                got = r, w = mine;
            } catch (Stop) {
            }
        }
        if (ended == 64) return got;
        if (ended) fail("lanes part");
        known.push_back(pending);
    }
}

int num(char**& a) { return atoi(*a++); }

int main(int, char** a) {
    ++a;
    DecodeParams p{};
    const int bm = num(a), wgs = num(a);
    p.H = num(a), p.delta = num(a), p.max_seq_len = num(a), p.fit_runs = num(a), p.line_weight = num(a), p.offsets_i64 = num(a), p.B = num(a);
    std::vector<int64_t> off64(1);
    for (int b = 0; b < p.B; ++b) off64.push_back(off64.back() + num(a));
    std::vector<int> off32(off64.begin(), off64.end());
    p.offsets = p.offsets_i64 ? (const void*)off64.data() : off32.data();
    p.num_mb = (p.delta + bm - 1) / bm, p.mb_magic = p.num_mb;
    p.line_wgs = (p.fit_runs * p.H + 7) / 8 * p.num_mb;
    const int slots = p.line_wgs * (p.line_weight ? p.B : 1), plane_slots = p.fit_runs + (p.line_weight ? p.B : 0);
    std::map<std::tuple<int, int, int>, std::map<int, Work>> made;
    std::set<int> used;
    long items = 0;
    for (int xcd = 0; xcd < 8; ++xcd)
        for (int lw = 0; lw < wgs; ++lw)  // the kernels' workgroups: their items by round, up to the first that decodes to nothing
            for (int round = 0, slot = lw; slot < slots; ++round, slot = round * wgs + (round & 1 ? wgs - 1 - lw : lw)) {
                Work w;
                int mb = -1;
                int64_t s0, s1;
                auto decode = [&](Work& m) {
                    return p.line_weight ? (bm == 256 ? decode_line<256, 64>(m, p, slot, xcd, s0, s1, mb) : decode_line<128, 64>(m, p, slot, xcd, s0, s1, mb))
                                         : (bm == 256 ? decode_fitted<256, 64>(m, p, slot, xcd, s0, s1, mb) : decode_fitted<128, 64>(m, p, slot, xcd, s0, s1, mb));
                };
                if (!wave(decode, w)) break;
                ++items;
                if (s0 != off64[w.b] || s1 != off64[w.b + 1] || w.jt_end <= w.jt_begin) fail("bounds");
                if (!made[{w.b, w.h, mb}].emplace(w.split, w).second) fail("a run twice");
                if (w.fit_slot >= 0 && (w.fit_slot >= p.H * p.num_mb * plane_slots || !used.insert(w.fit_slot).second)) fail("slot");
            }
    for (int b = 0; b < p.B; ++b)
        for (int h = 0; h < p.H; ++h)
            for (int mb = 0; mb < p.num_mb; ++mb) {
                const int64_t len = off64[b + 1] - off64[b], n = len < p.max_seq_len ? len : p.max_seq_len;
                const int end = (mb + 1) * bm < p.delta ? (mb + 1) * bm : p.delta;
                const int tiles = n > 0 && n >= p.delta ? (int)((n - p.delta + end + 63) / 64) : 0;
                const auto& runs = made[{b, h, mb}];
                int done = 0, split = 0;
                for (const auto& [s, w] : runs) {  // (in order: each continues the one before, and knows their number and the first one's partial sums)
                    if (s != split++ || w.jt_begin != done || (w.nsplit & 0xffff) != (int)runs.size()) fail("a run");
                    if (w.fit_slot != (runs.size() > 1 ? (h * p.num_mb + mb) * plane_slots + (w.nsplit >> 16) + s : -1)) fail("partial sums");
                    done = w.jt_end;
                }
                if (done != tiles) fail("tiles");
            }
    printf("%ld", items);
}
"""


@pytest.fixture(scope="module")
def decoded(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("needs g++")
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "generative-recommenders_amd", "csrc")
    text = open(os.path.join(csrc, "hstu_common.h")).read()
    source = text[text.index("// kv tiles of sequence `lane` for row block mb") : text.index("#define HSTU_PLAN_THREADS")]
    src = tmp_path_factory.mktemp("runs") / "runs.cpp"
    src.write_text(_HARNESS.replace("SOURCE", source))
    exe = src.with_suffix("")
    subprocess.run([gxx, "-O2", "-std=c++17", str(src), "-o", str(exe)], check=True)

    def run(bm, wgs, heads, delta, longest, runs, weight, i64, lengths):
        args = [bm, wgs, heads, delta, longest, runs, weight, int(i64), len(lengths), *lengths]
        proc = subprocess.run([str(exe)] + [str(x) for x in args], capture_output=True, text=True)
        assert proc.returncode == 0, (proc.stdout, args)
        return int(proc.stdout)

    return run


# lengths, heads, delta, rows of a row block, runs per plane: tiles exactly once whatever the number of runs -- one, as many as fit the chip, more than tiles; sequences without rows, shorter than
# the candidates, without history; one sequence and 64; a length above max_seq_len
SHAPES = [
    ([900], 1, 1, 128, 14), ([900], 3, 1, 128, 1), ([2000 + 37 * i for i in range(18)], 8, 3, 128, 64), ([133] * 32 + [4000] * 32, 4, 33, 128, 64),
    ([300, 8000] + [3640] * 30 + [4096, 301], 2, 300, 256, 64), ([500 + 331 * i for i in range(20)], 8, 129, 128, 32), ([0, 64, 7000, 20, 0, 513], 3, 64, 128, 40),
    ([10, 63], 2, 64, 128, 5), ([64], 1, 64, 256, 64), ([2**14 + 5, 100], 2, 37, 128, 30), ([129, 2500], 2, 129, 128, 128),
]


@pytest.mark.parametrize("lengths,heads,delta,bm,runs", SHAPES)
@pytest.mark.parametrize("weight", [4, 8])
def test_a_line_makes_every_tile_once(decoded, lengths, heads, delta, bm, runs, weight):
    longest = min(max(lengths), 2**14)
    wgs = (runs * heads + 7) // 8 * -(-delta // bm)
    got = [decoded(bm, wgs, heads, delta, longest, runs, weight, i64, lengths) for i64 in (False, True)]
    assert got[0] == got[1] and (got[0] > 0) == any(n >= delta for n in lengths if n)


@pytest.mark.parametrize("lengths,heads,delta,bm,runs", [s for s in SHAPES if s[4] >= 2 * len(s[0])])
def test_fitted_runs_make_every_tile_once(decoded, lengths, heads, delta, bm, runs):
    longest = min(max(lengths), 2**14)
    wgs = (runs * heads + 7) // 8 * -(-delta // bm)
    assert decoded(bm, wgs, heads, delta, longest, runs, 0, True, lengths) == decoded(bm, wgs, heads, delta, longest, runs, 0, False, lengths)
