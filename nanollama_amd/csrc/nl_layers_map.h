// nl_layers_map.h -- where the regions of nl_layers.h's exchange buffer lie, in 16-byte granules (plain C++: a test compiles it by itself).
//
// Every region begins a 128-byte line, and so does every XCD's copy: the vectors are written through by whichever XCD computed a part of them, a copy stays
// dirty in the L2 of its own, and a line of both would leave it to the caches whose bytes of it a later read sees.
#pragma once

namespace nl {

constexpr int LY_REC = 22;                 // granules of an attention record: max, sum, 64 values
constexpr int LY_HG = 3;                   // granules of half a tile
constexpr int LY_TG = 6;                   // ... of a tile
constexpr int LY_XCDS = 8;
constexpr int LY_LINE = 8;                 // granules of a cache line

struct LayersMap {
    int gq, gr, go, gp, gh, gx;            // q|k|v tiles; records [heads][rec_max][LY_REC]; the heads' outputs; x' half tiles; h tiles; x half tiles
    int loc, loc_n;                        // [LY_XCDS] copies of gp | gh | gx, `loc_n` apart
    int tickets;                           // [LY_XCDS] words, a line each
    int total;
};
constexpr LayersMap layers_map(int t_qkv, int heads, int rec_max, int t_d, int t_i) {
    LayersMap m{};
    int at = 0;
    auto take = [&at](int n) { const int first = at; at += (n + LY_LINE - 1) / LY_LINE * LY_LINE; return first; };
    m.gq = take(t_qkv * LY_TG); m.gr = take(heads * rec_max * LY_REC); m.go = take(heads * LY_REC);
    m.gp = take(t_d * 2 * LY_HG); m.gh = take(t_i * LY_TG); m.gx = take(t_d * 2 * LY_HG);
    m.loc = at;
    m.loc_n = (t_d * 4 * LY_HG + t_i * LY_TG + LY_LINE - 1) / LY_LINE * LY_LINE;
    take(LY_XCDS * m.loc_n);
    m.tickets = take(LY_XCDS * LY_LINE);
    m.total = at;
    return m;
}

}  // namespace nl
