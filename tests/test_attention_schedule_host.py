"""The order and split of the attention's work (csrc/fq_attention_schedule.hpp), compiled for the host: the search that every
workgroup makes for its own item hands out every piece of every workgroup once, longest first, within the grid of the launch."""
from __future__ import annotations

import ctypes
import os
import subprocess

import pytest

from tests import test_gpu_attention_rows as rows

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flashquant_amd", "csrc")

SOURCE = r"""
#include "fq_attention_schedule.hpp"
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <tuple>
#include <vector>
using namespace fq;

static int bad = 0;
#define CHECK(c, ...) do { if (!(c)) { if (++bad < 10) { printf(__VA_ARGS__); printf("\n"); } } } while (0)

struct Batch {
    std::vector<SeqShape> seqs;
    int G, D, H_KV, max_w;
    bool causal;
    SplitPlan plan;
    BatchWork work;
    int pieces(const SeqShape& s) const { return pieces_of(s, work, plan.split_w, plan.max_pieces, G, causal, D); }
    int count(int T) const {
        int c = 0;
        for (const auto& s : seqs) { const int n = pieces(s); c += n * (s.W - first_piece_with(s, T, n, G, causal)); }
        return c;
    }
    // as the kernel: (sequence, workgroup, piece, tile count of its class); sequence -1: none
    std::tuple<int, int, int, int> item(int place, bool ordered) const {
        int lo = 0, hi = 0x3fffffff, rem = place;
        if (ordered) {
            if (place >= count(0)) return {-1, 0, 0, 0};
            hi = 1;
            while (count(hi) > place) { lo = hi; hi *= 2; }
            while (hi - lo > 1) { const int mid = (lo + hi) >> 1; if (count(mid) > place) lo = mid; else hi = mid; }
            rem = place - count(hi);
        }
        for (size_t i = 0; i < seqs.size(); ++i) {
            const auto& s = seqs[i];
            const int n = pieces(s), x0 = first_piece_with(s, lo, n, G, causal);
            const int mine = n * (first_piece_with(s, hi, n, G, causal) - x0);
            if (rem < mine) return {int(i), x0 + rem / n, rem % n, lo};
            rem -= mine;
        }
        return {-1, 0, 0, 0};
    }
};

int main() {
    std::mt19937 rng(7);
    auto pick = [&](int lo, int hi) { return int(std::uniform_int_distribution<int>(lo, hi)(rng)); };
    int split_batches = 0, split_seqs = 0, whole_in_plan = 0;
    for (int round = 0; round < 1500; ++round) {
        Batch b;
        const int groups[] = {1, 2, 3, 4, 5, 8, 16}, heads[] = {1, 2, 4, 8, 32}, dims[] = {64, 128, 256};
        b.G = groups[pick(0, 6)];
        b.H_KV = heads[pick(0, 4)];
        b.D = dims[pick(0, 2)];
        b.causal = pick(0, 3) > 0;
        const int S = pick(1, round % 4 ? 12 : 90), longest = pick(0, 2) ? 300 : 3000, context = pick(0, 1) ? 300 : 9000;
        std::vector<int> nq(S), kv(S);
        int max_q = 1, max_kv = 1;
        int64_t total = 0;
        for (int s = 0; s < S; ++s) {
            nq[s] = pick(0, 3) ? (pick(0, 1) ? 1 : pick(0, longest)) : pick(0, 5);
            kv[s] = pick(0, 9) ? nq[s] + pick(0, context) : pick(0, 40);
            max_q = nq[s] > max_q ? nq[s] : max_q;
            max_kv = kv[s] > max_kv ? kv[s] : max_kv;
            total += nq[s];
        }
        const int64_t table = max_kv + int64_t(pick(0, 2)) * 4096;                 // the host knows the block table only
        b.max_w = int(((int64_t(max_q) + 31) / 32 * b.G + 7) / 8);
        b.plan = plan_split(S, b.H_KV, b.max_w, (table + 63) / 64, 256, b.D, false);
        uint32_t tiles = 0, rows = 0;
        for (int s = 0; s < S; ++s) {
            const SeqShape sh = make_seq_shape(nq[s], kv[s], kv[s] > nq[s] ? kv[s] - nq[s] : 0, b.G, b.max_w);
            b.seqs.push_back(sh);
            for (int x = 0; x + 1 < sh.W; ++x)
                CHECK(tiles_of(sh, x, b.G, b.causal) <= tiles_of(sh, x + 1, b.G, b.causal), "tiles decrease with x");
            for (int T = 0; T <= sh.all_tiles + 2; ++T) {                           // against a search
                int x = 0;
                while (x < sh.W && tiles_of(sh, x, b.G, b.causal) < T) ++x;
                CHECK(first_with(sh, T, b.G, b.causal) == x, "first_with(%d) of %d queries, %d keys", T, nq[s], kv[s]);
            }
            if (sh.W > 0)
                tiles += uint32_t(sh.W) * uint32_t(tiles_of(sh, 0, b.G, b.causal) + tiles_of(sh, sh.W - 1, b.G, b.causal) + 1) / 2;
            if (sh.W <= b.plan.split_w) rows += uint32_t(sh.NQ) * uint32_t(b.G);
        }
        b.work = {share_of(tiles * uint32_t(b.H_KV), 256), int(rows * uint32_t(b.H_KV) >> 8)};
        int all = 0;
        for (const auto& s : b.seqs) {
            const int n = b.pieces(s);
            CHECK(n >= 1 && n <= (b.plan.max_pieces > 1 ? b.plan.max_pieces : 1), "%d pieces", n);
            CHECK(n == 1 || s.W <= b.plan.split_w, "a split sequence without slots");
            CHECK(n == 1 || may_split(s, b.plan.split_w, b.plan.max_pieces, b.G, b.causal, b.D), "split where may_split says no");
            all += n * s.W;
            split_seqs += n > 1;
            whole_in_plan += n == 1 && s.W > 0 && b.plan.max_pieces > 1;
        }
        split_batches += b.plan.max_pieces > 1;
        // the grid: as the host counts it, with and without the number of tokens
        int64_t places = int64_t(S) * b.max_w;
        const int64_t most = (total / 32 + S) * b.G / 8 + S;
        places = most < places ? most : places;
        const int64_t extra = int64_t(S) * b.plan.split_w * (b.plan.max_pieces - 1);
        CHECK(all <= places + extra, "%d items, %lld places", all, (long long)(places + extra));
        CHECK(b.plan.max_pieces < 2 || int64_t(S) * b.plan.split_w <= places + extra, "fewer workgroups than slots");
        for (bool ordered : {true, false}) {
            std::set<std::tuple<int, int, int>> seen;
            int last = 1 << 30;
            for (int place = 0; place < all; ++place) {
                const auto [seq, x, piece, T] = b.item(place, ordered);
                CHECK(seq >= 0 && seen.insert({seq, x, piece}).second, "place %d of %d: none or twice", place, all);
                if (seq < 0) break;
                CHECK(x >= 0 && x < b.seqs[seq].W && piece < b.pieces(b.seqs[seq]), "out of the sequence");
                CHECK(T <= last, "not longest first");
                last = T;
            }
            CHECK(int(seen.size()) == all, "%zu of %d items", seen.size(), all);
            CHECK(std::get<0>(b.item(all, ordered)) < 0 && std::get<0>(b.item(all + 100, ordered)) < 0, "work behind the end");
        }
    }
    CHECK(split_batches > 100 && split_seqs > 100 && whole_in_plan > 100, "too few splits tried: %d %d %d", split_batches, split_seqs, whole_in_plan);
    printf("%d wrong\n", bad);
    return bad != 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("schedule")
    (d / "schedule.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", f"-I{CSRC}", str(d / "schedule.cpp"), "-o", str(d / "schedule")], check=True)
    return str(d / "schedule")


def test_every_piece_is_handed_out_once(program):
    r = subprocess.run([program], stdout=subprocess.PIPE, text=True, timeout=300)
    assert r.returncode == 0, r.stdout


CONTIGUOUS = r"""
#include "fq_attention_expanded.hpp"
#include "fq_attention_schedule.hpp"
namespace fq_host { int device_cu_count() { return 256; } }
using namespace fq;
// whether the operator, with room for all that it asks for, runs such a call on expanded keys instead
extern "C" int expanded(int B, int HQ, int HKV, int NQ, int NKV, int D, int is_causal) {
    return plan_expanded(B, HKV, NQ, NKV, HQ / HKV, D, is_causal && NQ > 1).per_chunk > 0;
}
// pieces of a call over contiguous keys on 256 CUs, as its entry works them out; + 100: whole prompts' combine launch
extern "C" int pieces(int B, int HQ, int HKV, int NQ, int NKV, int D, int is_causal) {
    const int G = HQ / HKV, max_w = ((NQ + 31) / 32 * G + 7) / 8;
    const bool causal = is_causal && NQ > 1;
    const int64_t keys = causal && NKV > NQ ? NQ : NKV;
    const SplitPlan sp = plan_split(B, HKV, max_w, (keys + 63) / 64, 256, D, causal);
    if (sp.max_pieces < 2) return 1;
    const SeqShape sh = make_seq_shape(NQ, NKV, 0, G, max_w);
    const uint32_t tiles = uint32_t(B * HKV) * (uint32_t(sh.W) * uint32_t(tiles_of(sh, 0, G, causal) + tiles_of(sh, sh.W - 1, G, causal) + 1) / 2);
    const int rows = sh.W <= sp.split_w ? B * NQ * HQ : 0;
    const int n = pieces_of(sh, {share_of(tiles, 256), rows >> 8}, sp.split_w, sp.max_pieces, G, causal, D);
    return n < 2 ? 1 : n + (sp.split_w > 1 && 2 * B * HKV * sp.split_w >= 256 ? 100 : 0);
}
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    d = tmp_path_factory.mktemp("pieces")
    (d / "pieces.cpp").write_text(CONTIGUOUS)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", str(d / "pieces.cpp"), "-o", str(d / "pieces.so")], check=True)
    return ctypes.CDLL(str(d / "pieces.so"))


def test_the_gpu_tests_reach_what_they_name(library):
    """The cases of the tests on contexts in pieces run in pieces, and through the combine launch that they are there for: as the
    operator runs them, or (causal prompts, which have room for expanded keys there) with room for pieces alone."""
    pieces, expanded = library.pieces, library.expanded
    assert all(pieces(*c, 0) > 1 for c in rows.SPLIT) and all(pieces(*c, 0) == 1 for c in rows.NOT_SPLIT)
    assert not any(expanded(*c, 0) for c in rows.SPLIT + rows.NOT_SPLIT)
    for shortest in ((1, 8, 2, 1, 449, 128), (1, 4, 1, 3, 705, 64), (1, 8, 1, 2, 449, 256)):
        assert shortest in rows.SPLIT and pieces(*shortest[:4], shortest[4] - 1, shortest[5], 0) == 1
    for d in (64, 128, 256):
        for c in rows.IN_PIECES:
            assert (pieces(*c, d, 0) > 100) == (c[3] == 390) and pieces(*c, d, 0) > 1 and not expanded(*c, d, 0), (c, d)
        for c in rows.WHOLE_PROMPTS:
            assert pieces(*c[:5], d, int(c[5])) > 100 and bool(expanded(*c[:5], d, int(c[5]))) == c[5], (c, d)
        assert pieces(1, 8, 1, 4201, 4201, d, 1) > 100 and expanded(1, 8, 1, 4201, 4201, d, 1)
    assert {pieces(*c[:5], 256, int(c[5])) > 1 for c in rows.WIDE if not expanded(*c[:5], 256, int(c[5]))} == {True, False}
