// Work lists of plans over random block structures: the lists the library
// builds pass its own check, and a wrong chunk, step, step count, slot, tile or
// reduction does not.
#include <cstdio>
#include <functional>
#include <random>

#include "errors.hpp"
#include "pivot.hpp"

using namespace vmps;

static int errors = 0;
static void expect(bool ok, const char* what, const char* detail = "") {
  if (!ok) {
    ++errors;
    std::printf("FAILED: %s %s\n", what, detail);
  }
}

// sectors of the left bond (rows) and of the right one (columns): every vector
// block L_i x R_j, every X and Z between neighbouring sectors
static TripleSet triples(const std::vector<int64_t>& left, const std::vector<int64_t>& right) {
  TripleSet S;
  const int nl = (int)left.size(), nr = (int)right.size();
  for (int i = 0; i < nl; ++i)
    for (int j = 0; j < nr; ++j) {
      S.Yb.push_back({S.ysize, left[i], right[j]});
      S.ysize += left[i] * right[j];
    }
  S.Ob = S.Yb;
  S.osize = S.ysize;
  std::vector<std::vector<int>> x(nl, std::vector<int>(nl, -1)), z(nr, std::vector<int>(nr, -1));
  auto add = [](std::vector<BlockDim>& b, int64_t& size, int64_t r, int64_t c) {
    b.push_back({size, r, c});
    size += r * c;
    return (int)b.size() - 1;
  };
  for (int o = 0; o < nl; ++o)
    for (int i = 0; i < nl; ++i)
      if (std::abs(o - i) <= 1) x[o][i] = add(S.Xb, S.Xsize, left[o], left[i]);
  for (int i = 0; i < nr; ++i)
    for (int o = 0; o < nr; ++o)
      if (std::abs(o - i) <= 1) z[i][o] = add(S.Zb, S.Zsize, right[i], right[o]);
  S.Xgather.push_back({nullptr, 0, S.Xsize});  // sizes without data
  S.Zgather.push_back({nullptr, 0, S.Zsize});
  for (int oi = 0; oi < nl; ++oi)
    for (int oj = 0; oj < nr; ++oj)
      for (int ii = 0; ii < nl; ++ii)
        for (int ij = 0; ij < nr; ++ij)
          if (x[oi][ii] >= 0 && z[ij][oj] >= 0) {
            Term t{};
            t.out_v = oi * nr + oj;
            t.l_blk = x[oi][ii];
            t.in_v = ii * nr + ij;
            t.r_blk = z[ij][oj];
            t.c = 0.5;
            S.terms.push_back(t);
          }
  return S;
}

struct Lists {
  std::vector<TileC> tiles;
  std::vector<ChunkC> chunks;
  int64_t kstep;
  std::vector<BigItemC> items;
  std::vector<BigRedC> reds;
  int64_t slots;
  bool ok() const {
    try {
      check_big_items(tiles, chunks, kstep, items, reds, slots);
      return true;
    } catch (const VmpsError&) {
      return false;
    }
  }
};

static void corrupt(const Lists& good) {
  auto refused = [&](const char* what, const std::function<bool(Lists&)>& f) {
    Lists bad = good;
    if (f(bad)) expect(!bad.ok(), "refused:", what);
  };
  size_t w = 0, whole = good.items.size();
  for (size_t i = 0; i < good.items.size(); ++i) {
    if (good.items[i].tile >= 0) w = i;
    if (good.items[i].tile >= 0 && good.items[i].slot < 0 && good.items[i].nsteps > 0) whole = i;
  }
  refused("tile", [&](Lists& b) { b.items[w].tile = (int32_t)b.tiles.size(); return true; });
  refused("chunk past the tile's", [&](Lists& b) { b.items[w].chunk = b.tiles[b.items[w].tile].chunk_end; return true; });
  refused("chunk before the tile's", [&](Lists& b) { b.items[w].chunk = b.tiles[b.items[w].tile].chunk_begin - 1; return true; });
  refused("step", [&](Lists& b) { b.items[w].step += 1 << 20; return true; });
  refused("negative step", [&](Lists& b) { b.items[w].step = -1; return true; });
  refused("one step more", [&](Lists& b) { ++b.items[w].nsteps; return true; });
  refused("one step less", [&](Lists& b) { --b.items[w].nsteps; return true; });
  refused("item dropped", [&](Lists& b) { b.items[w].tile = -1; return true; });
  refused("item twice", [&](Lists& b) { b.items.push_back(b.items[w]); return true; });
  refused("whole tile into a slot", [&](Lists& b) { if (whole >= b.items.size()) return false; b.items[whole].slot = b.slots; return true; });
  if (good.reds.empty()) return;
  size_t part = 0, other = 0;
  for (size_t i = 0; i < good.items.size(); ++i)
    if (good.items[i].tile >= 0 && good.items[i].slot >= 0) other = part, part = i;
  refused("slot past the last", [&](Lists& b) { b.items[part].slot = b.slots; return true; });
  refused("slot shared", [&](Lists& b) { b.items[part].slot = b.items[other].slot; return true; });
  refused("part stored as the tile", [&](Lists& b) { b.items[part].slot = -1; return true; });
  refused("fewer slots", [&](Lists& b) { --b.slots; return true; });
  refused("reduction dropped", [&](Lists& b) { b.reds.pop_back(); return true; });
  refused("reduction twice", [&](Lists& b) { b.reds.push_back(b.reds[0]); return true; });
  refused("reduction of too few parts", [&](Lists& b) { --b.reds[0].nsplit; return true; });
  refused("reduction into another tile", [&](Lists& b) { b.reds[0].tile = (b.reds[0].tile + 1) % (int32_t)b.tiles.size(); return b.tiles.size() > 1; });
  refused("reduction past the slots", [&](Lists& b) { b.reds.back().slot = b.slots; return true; });
}

// one large block row against a thin one: the same classes and work in the
// histogram, but only the first is dominated by large blocks
static void signatures() {
  HostPlan a, b;
  build_plan(triples({320}, {64}), a);
  build_plan(triples({400}, {33}), b);
  expect(a.large && !b.large, "one plan of each kind");
  expect(tile_signature(a) != tile_signature(b), "plans of different rules have different signatures");
}

// the widths of the LDS tiles change at 256 tiles of 128 x 128 in blocks of 128 and more
static void widths() {
  for (int64_t n : {255, 256}) {
    HostPlan H;
    build_plan(triples({128}, {128 * n}), H);
    expect(H.big_min64 > 0 && H.big_edge == (n < 256 ? 64 : 128), "edge of the FP64 / FP32 tiles");
    for (bool xu : {false, true}) {
      H.explicit_u = xu;
      build_tiles(H);
      Bf16Layout B;
      build_bf16_layout(H, B);
      expect(B.wideC == (xu && n >= 256), "width of the split-BF16 stage C tiles");
    }
  }
  // a pivot of the size that the 128-wide kernels are tested with: tiles cut along K
  HostPlan H;
  build_plan(triples({641, 700, 736, 765}, {769, 595, 935, 1020}), H);
  Bf16Layout B;
  build_bf16_layout(H, B);
  expect(H.big_edge == 128 && !H.redsC_b.empty(), "128-wide tiles cut along K");
  expect(B.wideC && !B.redsC.empty(), "128 x 256 tiles cut along K");
}

int main() {
  signatures();
  widths();
  std::mt19937 rng(5);
  int split = 0, edge128 = 0, wide = 0;
  const std::vector<std::vector<int64_t>> bonds = {{1, 17, 64, 65, 130}, {3, 260, 31, 127}, {300, 5, 257}, {640, 29},
                                                   {1200, 1100, 900}, {1400, 1023, 1}};
  for (const auto& left : bonds)
    for (bool xu : {false, true})
      for (int min64 : {1, 33, 128}) {
        const auto& right = bonds[rng() % bonds.size()];
        HostPlan H;
        const TripleSet S = triples(left, right);
        build_plan(S, H);
        H.explicit_u = xu;
        H.big_min = min64;
        build_tiles(H);
        set_wave_edge(H, 32, min64);  // throws if a list is wrong
        Bf16Layout B;
        build_bf16_layout(H, B);
        const Lists f{H.tilesC_b, H.chunksC, kBigKd, H.itemsC_b, H.redsC_b, H.slotsC_b};
        const Lists b{B.tilesC_big, H.chunksC, kBigK, B.itemsC, B.redsC, B.slotsC};
        for (const Lists* l : {&f, &b}) {
          expect(l->ok(), "the library's own lists");
          if (!l->tiles.empty()) corrupt(*l);
          split += !l->reds.empty();
        }
        edge128 += H.big_edge == 128;
        wide += B.wideC;
      }
  expect(split > 0 && edge128 > 0 && wide > 0, "every kind of list was built");
  std::printf("%d errors; lists with split tiles %d, 128 wide %d, 128 x 256 %d\n", errors, split, edge128, wide);
  return errors ? 1 : 0;
}
