"""Which attention calls run on keys and values expanded once (csrc/fq_attention_expanded.hpp), compiled for the host."""
from __future__ import annotations

import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flashquant_amd", "csrc")

SOURCE = r"""
#include "fq_attention_expanded.hpp"
namespace fq_host { int device_cu_count() { return 256; } }
using namespace fq;
extern "C" int paged(int64_t seqs, int64_t total_q, int64_t max_q, int64_t max_kv, int HQ, int HKV, int D) {
    return plan_expanded_paged(seqs, total_q, max_q, max_kv, HKV, HQ / HKV, D).per_chunk > 0;
}
extern "C" int contiguous(int64_t batch, int HQ, int HKV, int64_t n_q, int64_t n_kv, int D, int causal) {
    return plan_expanded(batch, HKV, n_q, n_kv, HQ / HKV, D, causal != 0).per_chunk > 0;
}
// pieces of a workgroup over keys without a mask at 256 coordinates, by the rule of the launch
extern "C" int pieces(int workgroups, int tiles) {
    const int64_t share = (int64_t(workgroups) * tiles + 255) / 256;
    int best_k = 1;
    int64_t best = 0;
    for (int i = 0; i < kPieceChoices; ++i) {
        const int64_t piece = piece_choice(i, tiles, 2 * kPieceTiles), k = (tiles + piece - 1) / piece;
        const int64_t ns = batch_ns(piece, share, workgroups * k, k > 1 ? workgroups * k : 0, 256, 256, true);
        if (i == 0 || 20 * ns < 19 * best) {
            best = ns;
            best_k = int(k);
        }
    }
    return best_k;
}
extern "C" int64_t share(int64_t workgroups, int first, int last, int H_KV, int places) {
    return share_of_work(work_of(workgroups, first, last), H_KV, places);
}
// against workgroups and their tiles counted one by one; how many differ
extern "C" int counted(int n_q, int n_kv, int G, int D, int causal) {
    const int TS = D == 256 ? 5 : 6, units = (n_q + 31) / 32 * G, W = (units + 3) / 4, keys = causal && n_kv > n_q ? n_q : n_kv;
    const int tiles = (keys + (1 << TS) - 1) >> TS;
    const ContiguousWork work{W, tiles, (1 << TS) / 32 * G, causal != 0};
    auto tiles_of = [&](int x) {
        int pos = 32 * ((4 * x + 3 < units - 1 ? 4 * x + 3 : units - 1) / G) + 31;
        pos = pos < n_q - 1 ? pos : n_q - 1;
        return causal && (pos >> TS) + 1 < tiles ? (pos >> TS) + 1 : tiles;
    };
    int64_t all = 0;
    int wrong = tiles_of(W - 1) != tiles;
    for (int x = 0; x < W; ++x) all += tiles_of(x);
    wrong += all != work.all();
    for (int i = 0; i < kPieceChoices; ++i) {
        const int piece = piece_choice(i, tiles, kPieceTiles << (6 - TS));
        int64_t items = 0, split = 0;
        for (int x = 0; x < W; ++x) {
            const int k = (tiles_of(x) + piece - 1) / piece;
            items += k;
            split += k > 1 ? k : 0;
        }
        wrong += items != work.items(piece) || split != work.split(piece);
    }
    return wrong;
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    d = tmp_path_factory.mktemp("plans")
    (d / "plans.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-shared", "-fPIC", f"-I{CSRC}", str(d / "plans.cpp"), "-o", str(d / "plans.so")], check=True)
    return ctypes.CDLL(str(d / "plans.so"))


# (sequences, tokens, most of a sequence, columns of the block table in tokens, query heads, KV heads, dimension), and whether expanding
# is the faster way (measured): few rows of 128 coordinates on the keys of many pairs, several rounds of workgroups of the other kernel,
# rows that fill its workgroups, the other dimensions
PAGED = [((12, 12 * 214, 214, 224, 16, 16, 128), False), ((13, 13 * 83, 83, 96, 16, 16, 128), False), ((24, 24 * 150, 150, 160, 8, 8, 128), False), ((4, 4 * 300, 300, 304, 32, 32, 128), False),
         ((16, 16 * 16, 16, 16, 32, 8, 128), False), ((57, 57 * 17, 17, 32, 32, 4, 128), False),
         ((13, 980, 168, 288, 32, 16, 128), False),
         ((8, 8, 1, 16, 64, 8, 128), True), ((2, 426, 252, 256, 4, 4, 128), True), ((24, 24 * 150, 150, 160, 32, 32, 128), True),
         ((36, 141, 6, 16, 32, 8, 128), True), ((2, 20, 10, 16, 8, 8, 128), True),
         ((12, 10558, 2048, 4816, 32, 8, 128), True), ((12, 12 * 214, 214, 224, 16, 16, 256), True), ((1, 8192, 8192, 8192, 32, 8, 64), True)]


@pytest.mark.parametrize("sizes,expanded", PAGED)
def test_paged_batches_run_where_they_are_faster(plans, sizes, expanded):
    i64 = ctypes.c_int64
    assert bool(plans.paged(*(i64(n) for n in sizes[:4]), *sizes[4:])) == expanded


# (batch, query heads, KV heads, queries, keys, dimension, causal)
CONTIGUOUS = [((7, 16, 16, 20, 20, 128, 1), False), ((3, 32, 32, 28, 28, 128, 1), False), ((31, 4, 4, 17, 30, 128, 0), False), ((4, 32, 32, 300, 300, 128, 1), False),
              ((4, 32, 8, 65, 65, 64, 1), False), ((1, 32, 8, 33, 8000, 128, 0), False),
              ((3, 16, 16, 20, 20, 128, 1), True), ((4, 32, 32, 700, 700, 128, 1), True), ((1, 32, 8, 40, 40, 128, 1), True), ((7, 16, 16, 20, 20, 256, 1), True)]


@pytest.mark.parametrize("sizes,expanded", CONTIGUOUS)
def test_contiguous_calls_run_where_they_are_faster(plans, sizes, expanded):
    b, hq, hkv, nq, nkv, d, causal = sizes
    i64 = ctypes.c_int64
    assert bool(plans.contiguous(i64(b), hq, hkv, i64(nq), i64(nkv), d, causal)) == expanded


# (workgroups, tiles of 32 keys, pieces): 166 workgroups in two pieces are two rounds of 256 CUs, as long as one whole, in three still two
@pytest.mark.parametrize("workgroups,tiles,pieces", [(166, 383, 3), (150, 227, 3), (128, 200, 2), (250, 125, 1), (256, 300, 1), (20, 300, 12)])
def test_pieces_of_one_length_fill_their_rounds(plans, workgroups, tiles, pieces):
    assert plans.pieces(workgroups, tiles) == pieces


def test_the_share_of_large_batches(plans):
    """Workgroups times tiles go beyond 32 bits: 3 * 10^5 queries over 8 * 10^6 keys on one KV head, 16 query heads."""
    f = plans.share
    f.restype, f.argtypes = ctypes.c_int64, [ctypes.c_int64] + [ctypes.c_int] * 4
    for w, first, last, hkv in ((37500, 120000, 125000, 1), (1 << 20, 1, 1 << 18, 1), (1 << 20, 1 << 18, 1 << 18, 8), (3, 1, 4, 5)):
        assert f(w, first, last, hkv, 512) == (((w * (first + last) + 1) // 2) * hkv + 511) // 512


def test_workgroups_and_pieces_are_counted_right(plans):
    sizes = [(nq, nkv) for nq in (17, 31, 32, 33, 64, 65, 100, 128, 129, 1000, 3001, 4096, 5003) for nkv in (1, 31, 33, 64, 65, 129, nq - 1, nq, nq + 1, 2 * nq + 7)]
    for nq, nkv in sizes:
        for g in (1, 2, 3, 4, 5, 8, 12, 32):
            for d in (64, 128, 256):
                for causal in (0, 1):
                    assert plans.counted(nq, nkv, g, d, causal) == 0, (nq, nkv, g, d, causal)
