// Host emulation of the boundaries and walks of the fused parse and decode
// (k_fused_setup + k_fused_decode in szp_amd/csrc/szp_kernels.hip): sync_walk
// and fused_walk are the szp_geom.h functions the kernel calls; this file
// replays the kernel's glue tile by tile, with the byte buffer and the bitmap
// at their exact sizes so that AddressSanitizer catches any access outside
// them.  For each stream it compares the block positions with a plain serial
// walk of the chunks, and the stream-error verdict with the serial walk's.
//   fused_check <list>   lines: "<file> <n> <B> <T> <fastMode>"
// (the stream length is the file size, which may exceed the real stream).
// Geometries the fused kernel does not serve are skipped.
#include <stdio.h>
#include <stdlib.h>
#include <stdint.h>
#include <string.h>
#include <algorithm>
#include <memory>
#include <vector>

#include "szp_geom.h"

using namespace szp_amd;

static uint64_t rd64(const uint8_t *p)
{
    uint64_t v;
    memcpy(&v, p, 8);
    return v;
}

struct Result {
    bool bad = false;
    std::vector<uint64_t> pos;     // block positions, chunk-major
    std::vector<uint8_t> written;  // times each position was written
};

// Serial walk: the positions of every chunk's blocks and whether the stream
// passes the same validity rules the kernel enforces (chunk offsets in range,
// width bytes <= 32 on the chain, last block ending at the chunk end, or
// inside the buffer for the last chunk).
static Result serial_parse(const uint8_t *st, uint64_t len, const Geom &g)
{
    Result r;
    const uint64_t nblocks = (uint64_t)(g.T - 1) * g.nb0 + g.nblast;
    r.pos.assign(nblocks, ~0ull);
    if (len < g.body) {
        r.bad = true;
        return r;
    }
    for (uint32_t t = 0; t < g.T; ++t) {
        const uint64_t nt = chunk_len(g, t);
        const uint64_t off = rd64(st + 4 + 8ull * t);
        const uint64_t cs = g.body + off;
        if (nt == 0) {
            if (off != 0) r.bad = true;
            continue;
        }
        const uint64_t ce = (t + 1 < g.T) ? g.body + rd64(st + 4 + 8ull * (t + 1)) : len;
        if (off > len || cs + 4 > ce || ce > len) {
            r.bad = true;
            return r;
        }
        const uint64_t nb = (t == g.T - 1) ? g.nblast : g.nb0;
        if (g.mode == 2) {
            // Units: [q i32][width byte][...]; a one-value unit's width byte
            // is not read.
            uint64_t p = cs;
            if (cs + 5 > ce) {
                r.bad = true;
                return r;
            }
            for (uint64_t j = 0; j < nb; ++j) {
                if (p + 4 >= len || p >= ce) {
                    r.bad = true;
                    return r;
                }
                const uint64_t L = ((j + 1 < nb) ? g.B : nt - (nb - 1) * (uint64_t)g.B) - 1;
                const uint32_t b = st[p + 4];
                if ((L || j + 1 < nb) && b > 32) {
                    r.bad = true;
                    return r;
                }
                r.pos[(uint64_t)t * g.nb0 + j] = p;
                p += 4 + block_bytes(L ? b : 0, (uint32_t)L);
            }
            if (nb && (t + 1 < g.T ? p != ce : p > len)) {
                r.bad = true;
                return r;
            }
            continue;
        }
        uint64_t p = cs + 4;
        for (uint64_t j = 0; j < nb; ++j) {
            if (p >= ce) {
                r.bad = true;
                return r;
            }
            const uint32_t b = st[p];
            if (b > 32) {
                r.bad = true;
                return r;
            }
            r.pos[(uint64_t)t * g.nb0 + j] = p;
            const uint64_t L = (j + 1 < nb) ? g.B : (nt - 1) - (nb - 1) * (uint64_t)g.B;
            p += block_bytes(b, (uint32_t)L);
        }
        if (nb && (t + 1 < g.T ? p != ce : p > len)) {
            r.bad = true;
            return r;
        }
    }
    return r;
}

static uint64_t g_tiles = 0, g_sync = 0;

template <int MODE>
static Result emulate_mode(const uint8_t *st, uint64_t len, const Geom &g, bool &served)
{
    Result r;
    FusedShape f;
    served = fused_shape(g, len, &f);
    if (!served) return r;
    const uint64_t nblocks = (uint64_t)(g.T - 1) * g.nb0 + g.nblast;
    r.pos.assign(nblocks, ~0ull);
    r.written.assign(nblocks, 0);
    const uint32_t B = g.B, mode = MODE, S = f.S;

    // k_fused_setup
    std::vector<uint64_t> cstart(g.T), aend(g.T), ttab(g.T + 1);
    uint64_t tiles = 0;
    bool bad = len < g.body;
    for (uint32_t t = 0; t < g.T && !bad; ++t) {
        const uint64_t nt = chunk_len(g, t);
        const uint64_t off = rd64(st + 4 + 8ull * t);
        const uint64_t cs = g.body + off;
        ttab[t] = tiles;
        cstart[t] = aend[t] = cs;
        if (nt == 0) {
            if (off != 0) bad = true;
            continue;
        }
        const uint64_t nxt = (t + 1 < g.T) ? rd64(st + 4 + 8ull * (t + 1)) : 0;
        const uint64_t ce = (t + 1 < g.T) ? g.body + nxt : len;
        const uint64_t a0 = mode == 2 ? cs : cs + 4;
        if (off > len || nxt > len || a0 + (mode == 2 ? 5 : 0) > ce || a0 > ce || ce > len) {
            bad = true;
            break;
        }
        aend[t] = ce;
        const uint64_t nb = (t == g.T - 1) ? g.nblast : g.nb0;
        const uint64_t alen = ce - a0;
        if (nb && !alen) bad = true;
        tiles += nb && alen ? (alen + S - 1) / S : 1;
    }
    if (bad) {
        r.bad = true;
        return r;
    }
    ttab[g.T] = tiles;
    if (tiles > len / S + 1 + g.T) {
        fprintf(stderr, "more tiles than the launch has workgroups\n");
        exit(2);
    }
    std::vector<uint64_t> exit_st(tiles + 1, ~0ull), cnt_incl(tiles + 1, 0);
    const uint32_t nbuf = fused_buf_bytes(f), nword = fused_bitmap_words(f);

    for (uint64_t gt = 0; gt < tiles; ++gt) {
        ++g_tiles;
        uint32_t t = 0;
        while (t + 1 < g.T && ttab[t + 1] <= gt) ++t;
        const uint64_t i = gt - ttab[t];
        const bool first = i == 0;
        const uint64_t cs = cstart[t], ae = aend[t];
        const uint64_t s = cs + (mode == 2 ? 0 : 4) + i * S;
        const uint32_t span = (uint32_t)(std::min<uint64_t>(s + S, ae) - s);
        const uint64_t s0 = s & ~15ull;
        const uint32_t sh = (uint32_t)(s - s0);
        const uint64_t tl = std::min<uint64_t>(s + S + f.V + f.W + 16, len);
        const uint64_t nbt = (t == g.T - 1) ? g.nblast : g.nb0;
        std::unique_ptr<uint8_t[]> buf(new uint8_t[nbuf]);
        std::unique_ptr<uint32_t[]> bm(new uint32_t[nword]());
        memset(buf.get(), (int)(0xA5 + gt), nbuf);  // stale LDS contents
        for (uint64_t a = s0; a < tl; a += 16) {
            const uint64_t m = a + 16 <= len ? 16 : len - a;
            memcpy(buf.get() + (a - s0), st + a, m);
        }
        const uint8_t *tb = buf.get() + sh;

        std::vector<uint32_t> bnd(f.nsec + 1, kFusedNone);
        for (uint32_t b = 0; b <= f.nsec; ++b) {
            const uint32_t u = b == f.nsec ? S : b * f.sec;
            if (b == 0 && first) {
                bnd[b] = 0;
            } else if (s + u + f.V <= ae && s + u + f.V + 8 <= len) {
                std::vector<uint32_t> left;
                const uint32_t lanes = 1u << f.ll;
                for (uint32_t l = 0; l < lanes; ++l) {
                    const uint32_t c = std::min(u + f.per * l, u + f.W);
                    sync_walk<MODE>(tb, c, std::min(c + f.per, u + f.W), u + f.W - 1, u + 2 * f.W, f,
                                    [&](uint32_t p) {
                        if (p > u + 3 * f.W) exit(2);  // outside the bits that are taken back
                        if (std::find(left.begin(), left.end(), p) == left.end()) left.push_back(p);
                    });
                }
                if (left.size() > lanes) left.clear();
                for (uint32_t X = u + 2 * f.W;;) {
                    uint32_t least = kFusedNone, most = 0;
                    for (uint32_t p : left)
                        if (p != kFusedNone) least = std::min(least, p), most = std::max(most, p);
                    if (least == most) bnd[b] = least;
                    if (least >= most || X == u + f.V) break;
                    X = std::min(X + f.W, u + f.V);
                    for (uint32_t &p : left)
                        if (p != kFusedNone) p = sync_more<MODE>(tb, p, X, f);
                }
            }
        }
        g_sync += bnd[0] != kFusedNone;
        uint32_t brk = kFusedNone;
        for (uint32_t w = 0; w < f.nsec; ++w) {
            uint32_t p = bnd[w];
            bool broken = false;
            if (p == kFusedNone) {
                if (w) continue;
                const uint64_t e = exit_st[gt - 1];
                if (e == ~0ull) {
                    fprintf(stderr, "tile waits for an exit that is never published\n");
                    exit(2);
                }
                broken = e < s;
                p = broken ? 0 : (uint32_t)std::min<uint64_t>(e - s, S + f.W);
            }
            uint32_t end = kFusedNone;
            for (uint32_t k = w + 1; k <= f.nsec && end == kFusedNone; ++k) end = bnd[k];
            const bool open = end == kFusedNone;
            if (open) end = span;
            if (!broken) broken = !fused_walk<MODE>(tb, bm.get(), p, end, f);
            if (!open && p > end) broken = true;
            if (broken) brk = std::min(brk, std::min(p, end));
            if (open) exit_st[gt] = broken ? s + span : s + p;
        }
        const uint64_t pcnt = first ? 0 : cnt_incl[gt - 1];
        uint64_t cnt = 0, before = 0;
        uint64_t lastpos = ~0ull;
        for (uint32_t p = 0; p < nword * 32; ++p) {
            if (!bm_test(bm.get(), p)) continue;
            before += p < brk;
            const uint64_t bi = pcnt + cnt++;
            if (bi >= nbt) continue;
            r.pos[(uint64_t)t * g.nb0 + bi] = s + p;
            r.written[(uint64_t)t * g.nb0 + bi]++;
            if (bi == nbt - 1) lastpos = s + p;
            // The writing pass's width test.
            const uint64_t L = (bi == nbt - 1 ? chunk_len(g, t) - 1 - (nbt - 1) * (uint64_t)B
                                              : (mode == 2 ? B - 1 : B));
            const uint64_t q = s + p + (mode == 2 ? 4 : 0);
            const uint32_t b = q < tl ? st[q] : 255u;
            if (L && (b > 32 || q + block_bytes(b, (uint32_t)L) > tl)) r.bad = true;
        }
        cnt_incl[gt] = pcnt + cnt;
        if (brk != kFusedNone && pcnt + before < nbt) r.bad = true;
        if (gt + 1 == ttab[t + 1] && pcnt + cnt < nbt) r.bad = true;
        if (lastpos != ~0ull) {
            const uint64_t L = chunk_len(g, t) - 1 - (nbt - 1) * (uint64_t)B;
            const uint64_t q = lastpos + (mode == 2 ? 4 : 0);
            const uint32_t b = q < tl ? st[q] : 255u;
            const uint64_t e = q + block_bytes(b <= 32 && L ? b : 0, (uint32_t)L);
            if ((b > 32 && L) || (t + 1 < g.T ? e != ae : e > len)) r.bad = true;
        }
    }
    return r;
}

static Result emulate(const uint8_t *st, uint64_t len, const Geom &g, bool &served)
{
    return g.mode == 2 ? emulate_mode<2>(st, len, g, served) : emulate_mode<1>(st, len, g, served);
}

int main(int argc, char **argv)
{
    if (argc != 2) {
        fprintf(stderr, "usage: fused_check <case list>\n");
        return 2;
    }
    FILE *f = fopen(argv[1], "r");
    if (!f) return 2;
    char path[4096];
    unsigned long long n;
    int B, T, mode, ncase = 0, fail = 0, nbad = 0;
    while (fscanf(f, "%4095s %llu %d %d %d", path, &n, &B, &T, &mode) == 5) {
        FILE *sf = fopen(path, "rb");
        if (!sf) return 2;
        fseek(sf, 0, SEEK_END);
        const long len = ftell(sf);
        fseek(sf, 0, SEEK_SET);
        std::vector<uint8_t> st((size_t)len + 64, 0xEE);  // 64 bytes of slack: 16-byte loads
        if (fread(st.data(), 1, (size_t)len, sf) != (size_t)len) return 2;
        fclose(sf);
        Geom g;
        if (!make_geom(n, B, T, &g, 4, (uint32_t)mode)) {
            fprintf(stderr, "bad geometry %s\n", path);
            return 2;
        }
        bool served = false;
        const Result want = serial_parse(st.data(), (uint64_t)len, g);
        const Result got = emulate(st.data(), (uint64_t)len, g, served);
        if (!served) continue;
        ++ncase;
        nbad += want.bad;
        bool ok = want.bad == got.bad;
        if (ok && !want.bad) {
            for (size_t j = 0; j < want.pos.size(); ++j) {
                if (got.pos[j] != want.pos[j] || got.written[j] != 1) {
                    fprintf(stderr, "%s: block %zu at %llu, parsed %llu (written %d)\n", path, j,
                            (unsigned long long)want.pos[j], (unsigned long long)got.pos[j],
                            got.written[j]);
                    ok = false;
                    break;
                }
            }
        }
        if (!ok) {
            ++fail;
            fprintf(stderr, "FAIL %s n=%llu B=%d T=%d len=%ld serial_bad=%d parse_bad=%d\n", path,
                    n, B, T, len, (int)want.bad, (int)got.bad);
        }
    }
    fclose(f);
    printf("%d cases (%d invalid streams), %llu tiles (%llu with their own boundary), %d failures\n", ncase,
           nbad, (unsigned long long)g_tiles, (unsigned long long)g_sync, fail);
    return fail ? 1 : 0;
}
