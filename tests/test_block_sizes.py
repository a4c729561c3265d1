"""The device blocks the runtime keeps (csrc/pt_blocks.h, plain C++), on a
driver that counts: the size rule over the whole of size_t (it ends for every
size, rounds up by at most an eighth or to 512 bytes, and is stable), and what
is kept, given back and handed out again, out of memory included."""
import os
import subprocess

SIZES = r"""
#include "pt_blocks.h"
#include <initializer_list>
#include <stdio.h>
using pt::block_class;
static int check(size_t b)
{
    const size_t c = block_class(b);
    if (c < b || c % 512 || block_class(c) != c || (c - b >= 512 && c - b > b / 8)) {
        printf("%zu -> %zu\n", b, c);
        return 1;
    }
    return 0;
}
int main()
{
    int bad = 0;
    for (size_t b = 1; b < 100000; b++) bad += check(b);
    for (int s = 9; s < 63; s++)
        for (int k = -3; k <= 3; k++)
            for (size_t f = 8; f <= 16; f++) {
                const size_t b = ((size_t)f << s >> 3) + (size_t)(long long)k;
                if (b && b <= pt::kMaxBlockBytes) bad += check(b);
            }
    for (size_t b : {pt::kMaxBlockBytes, pt::kMaxBlockBytes - 1, pt::kMaxBlockBytes / 8 * 7}) bad += check(b);
    // above the largest request the rule is not asked, and ends all the same
    for (size_t b : {(size_t)1 << 63, SIZE_MAX, SIZE_MAX - 511}) block_class(b);
    return bad != 0;
}
"""


KEPT = r"""
#include "pt_blocks.h"
#include <assert.h>
#include <set>
#include <stdio.h>
struct Card {  // `room` bytes; streams are numbers, 0 the home stream
    std::unordered_map<void *, size_t> out;
    size_t used = 0, room = SIZE_MAX, calls = 0, waits = 0;
    uintptr_t next = 4096;
    std::set<int> captured;
    std::set<int> freed_on;
};
struct Driver {
    using Stream = int;
    using Status = int;
    static constexpr int kOk = 0, kNoMemory = 2;
    Card *card;
    int alloc(void **p, size_t n, int)
    {
        card->calls++;
        if (n > card->room - card->used) return kNoMemory;
        *p = (void *)card->next;
        card->next += n;
        card->used += n;
        card->out[*p] = n;
        return kOk;
    }
    int free(void *p, int s)
    {
        assert(card->out.count(p));
        card->used -= card->out[p];
        card->out.erase(p);
        card->freed_on.insert(s);
        return kOk;
    }
    void synchronize(int) { card->waits++; }
    bool capturing(int s) { return card->captured.count(s); }
};
using Blocks = pt::KeptBlocks<Driver>;
constexpr size_t MiB = 1 << 20;
static void *get(Blocks &k, size_t n, int s = 0)
{
    void *p = nullptr;
    assert(k.alloc(&p, n, s, 0) == 0);
    return p;
}
static void put(Blocks &k, void *p, int s = 0) { assert(k.release(p, s, 0) == 0); }
static void is(Blocks &k, size_t bytes, size_t blocks)
{
    size_t b, n;
    k.usage(&b, &n);
    if (b != bytes || n != blocks) fprintf(stderr, "%zu bytes in %zu blocks, not %zu in %zu\n", b, n, bytes, blocks);
    assert(b == bytes && n == blocks);
}
int main()
{
    {  // one block: taken again for its size only
        Card c;
        Blocks k(Driver{&c});
        void *p = get(k, 5 * MiB);
        is(k, 0, 0);
        put(k, p);
        is(k, 5 * MiB, 1);
        void *q = get(k, 4 * MiB);
        assert(q != p && c.calls == 2);
        assert(get(k, 5 * MiB - 1) == p && c.calls == 2);
        is(k, 0, 0);
        put(k, p);
        put(k, q);
        is(k, 9 * MiB, 2);
    }
    {  // other streams and captures pass by, in both directions
        Card c;
        Blocks k(Driver{&c});
        void *p = get(k, MiB);
        put(k, p, 1);
        is(k, 0, 0);
        assert(c.used == 0 && c.freed_on.count(1));
        p = get(k, MiB, 1);
        put(k, p);  // allocated elsewhere
        is(k, 0, 0);
        p = get(k, MiB);
        c.captured.insert(0);
        put(k, p);
        is(k, 0, 0);
        c.captured.clear();
        put(k, get(k, MiB));
        is(k, MiB, 1);
        assert(get(k, MiB, 1));
        c.captured.insert(0);
        assert(get(k, MiB));
        is(k, MiB, 1);
    }
    {  // what is kept, and the threshold on it and the blocks in use together
        Card c;
        Blocks k(Driver{&c});
        put(k, get(k, 5 * MiB));
        put(k, get(k, Blocks::kKeepBytes));
        is(k, Blocks::kKeepBytes, 1);
        put(k, get(k, Blocks::kKeepBytes + 1));
        is(k, Blocks::kKeepBytes, 1);
        k.set_threshold(6 * MiB, 0);
        is(k, 0, 0);
        void *p[6];
        for (auto &b : p) b = get(k, MiB);
        for (int i = 0; i < 6; i++) {
            put(k, p[i]);
            is(k, (i + 1) * MiB, i + 1);
        }
        void *two = get(k, 2 * MiB);  // 8 MiB with those kept
        is(k, 0, 0);
        assert(c.used == 2 * MiB);
        for (int i = 0; i < 5; i++) p[i] = get(k, MiB);  // 7 MiB in use
        put(k, p[0]);  // 6 with it
        is(k, 0, 0);
        put(k, p[1]);
        put(k, p[2]);
        is(k, 2 * MiB, 2);
        assert(c.used == 6 * MiB);
        void *big = get(k, 7 * MiB);
        is(k, 0, 0);
        put(k, p[3]);
        is(k, 0, 0);
        put(k, big);
        is(k, 0, 0);
        put(k, two);
        put(k, p[4]);
        is(k, 3 * MiB, 2);
        k.set_threshold(2 * MiB, 0);
        is(k, 0, 0);
        assert(c.used == 0);
        k.set_threshold(0, 0);
        put(k, get(k, 5 * MiB));
        is(k, 5 * MiB, 1);
    }
    for (int s = 0; s < 2; s++) {  // out of memory: what is kept makes room, once, and then the call fails
        Card c;
        Blocks k(Driver{&c});
        c.room = 64 * MiB;
        void *held = get(k, 8 * MiB);
        void *a = get(k, 24 * MiB), *b = get(k, 24 * MiB);
        put(k, a);
        put(k, b);
        is(k, 48 * MiB, 2);
        void *p = get(k, 40 * MiB, s);
        is(k, 0, 0);
        assert(c.waits == 1 && c.freed_on.size() == 1);
        put(k, p, s);
        is(k, 0, 0);
        // no room for the rounded size, room for the size itself: not kept
        if (s == 0) {
            const size_t n = 56 * MiB - 3 * MiB + 1;  // rounded up to 56 MiB, 8 are held
            c.room = 8 * MiB + n;
            p = get(k, n);
            assert(c.used == 8 * MiB + n);
            put(k, p);
            is(k, 0, 0);
        }
        void *none = nullptr;
        put(k, get(k, MiB));
        assert(k.alloc(&none, 65 * MiB, s, 0) == Driver::kNoMemory && !none);
        is(k, 0, 0);
        // within a capture nothing is given back, whichever stream it is on
        c.captured = {s};
        c.room = 64 * MiB;
        void *kept = nullptr;
        if (s == 1) {
            c.captured.clear();
            put(k, get(k, MiB));
            c.captured = {1};
            assert(k.alloc(&kept, 65 * MiB, 1, 0) == Driver::kNoMemory);
            c.captured = {0};
            assert(k.alloc(&kept, 65 * MiB, 1, 0) == Driver::kNoMemory);
            is(k, MiB, 1);
        } else {
            assert(k.alloc(&kept, 65 * MiB, 0, 0) == Driver::kNoMemory);
        }
        put(k, held, 1);
    }
    Card c;
    Blocks k(Driver{&c});
    void *p = nullptr;
    for (size_t n : {SIZE_MAX, (size_t)1 << 63}) assert(k.alloc(&p, n, 0, 0) == Driver::kNoMemory && c.calls == 0);
    return 0;
}
"""


def _run(tmp_path, program):
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "php-gpu-tensors_amd", "csrc")
    src, exe = tmp_path / "blocks.cpp", tmp_path / "blocks"
    src.write_text(program)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", csrc, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout + run.stderr


def test_rule(tmp_path):
    _run(tmp_path, SIZES)


def test_kept(tmp_path):
    _run(tmp_path, KEPT)
