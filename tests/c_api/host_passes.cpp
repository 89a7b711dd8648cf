// The planners against their kernels' limits, without a GPU: passes are
// planned from real decompositions through the library's own internal
// headers, and what a launch would ask for is checked here.
// Usage: host_passes <check>; prints OK.
#include <sys/resource.h>
#include <unistd.h>

#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "block_decomp.h"
#include "fft_program.h"

static int failures = 0;

// Packed blocks of shape over grid.
struct Layout {
  MPI_Comm comm;
  Decomp d;
  dm::HostLayout h;
  Layout(const std::vector<int> &shape, const std::vector<int> &grid) {
    int ranks = 1;
    for (int g : grid) ranks *= g;
    comm = dm_world_create(ranks);
    std::vector<DimDecomp> dims;
    for (size_t i = 0; i < shape.size(); i++) dims.push_back(makeBlockDecomp(shape[i], grid[i]));
    d = makePackedDecomp(comm, (int)shape.size(), dims.data());
    h = dm::layout_from_decomp(d);
  }
  ~Layout() {
    freeDecomp(d);
    dm_world_free(comm);
  }
  dm::Side side() const {
    i64 most = 1;
    for (i64 e : h.slot_extent) most = e > most ? e : most;
    return dm::make_side(h, most);
  }
};

// A workgroup's LDS, for every combination of line length, rank positions
// along the line and uneven sides; the middle axis makes a side uneven, the
// last axis the line stride (64 KiB or more with 130 points).
static void lds() {
  for (int n : {256, 360, 512, 729, 1000, 1024, 2048, 4096})
    for (int np : {1, 2, 6, 7, 16, 20, 32, 34, 47, 64, 68, 100, 128, 146, 256}) {
      if (np > n / 2) continue;
      const Layout even({n, 66, 130}, {1, 2, 1}), uneven({n, 65, 130}, {np, 2, 1}), local({n, 65, 130}, {1, 1, 1});
      const dm::Side e = local.side(), s = uneven.side();
      for (int form = 0; form < 3; form++)
        for (int dbl : {0, 1}) {
          dm::TableBuilder tb;
          dm::PendingPass pp;
          if (!dm::plan_pass(uneven.comm, form == 1 ? e : s, form == 0 ? e : s, 0, dbl, false, nullptr, nullptr, tb, &pp)) {
            printf("no pass: n %d np %d form %d dbl %d\n", n, np, form, dbl);
            failures++;
            continue;
          }
          const size_t need = dm::fft_lds_bytes(pp.L);
          if (need > 160 * 1024 || pp.L.T < 1) {
            printf("%zu bytes of LDS: n %d np %d form %d dbl %d T %d\n", need, n, np, form, dbl, pp.L.T);
            failures++;
          }
        }
    }
}

// Tables of a pass: within the 64 MiB that the line bases of uniform sides
// may take, however many rank positions a line crosses.
static void tables() {
  const Layout uneven({64, 2101, 128}, {1, 1100, 1}), local({64, 2101, 128}, {1, 1, 1});
  const dm::Side s = uneven.side(), e = local.side();
  for (int form = 0; form < 4; form++) {
    dm::TableBuilder tb;
    dm::PendingPass pp;
    if (!dm::plan_pass(uneven.comm, form & 1 ? e : s, form & 2 ? e : s, 1, 1, false, nullptr, nullptr, tb, &pp) ||
        tb.host.size() > (size_t)64 << 20) {
      printf("%zu bytes of tables, form %d\n", tb.host.size(), form);
      failures++;
    }
  }
}

// A reshape tile's LDS, for every element size, tile axis length, array size
// and number of rank positions that the owned kernels take.
static void reshape() {
  for (int bytes : {1, 2, 4, 8, 12, 16, 24})
    for (int la : {8, 16, 17, 64, 500})
      for (int lb : {8, 16, 17, 64, 500})
        for (int batch : {1, 100, 10000, 1000000})
          for (int pairs : {1, 100, dm::kReshapePairs})
            for (int form = 0; form < 8; form++) {
              dm::ReshapeLaunch L;
              memset(&L, 0, sizeof L);
              L.owned = 1;
              L.ndim = 3;
              L.L[0] = batch;
              L.L[1] = la;
              L.L[2] = lb;
              L.a = 1;
              L.b = 2;
              L.elem_bytes = bytes;
              L.src.uniform = form & 1;
              L.dst.uniform = form >> 1 & 1;
              L.below_4g = form >> 2 & 1;
              L.ss.np[0] = L.sd.np[1] = pairs;
              L.ss.np[1] = L.sd.np[0] = 1;
              const size_t need = dm::reshape_tile_lds(L);
              if (need == 0 || need > 64 * 1024) {
                printf("%zu bytes of LDS: %d bytes, %d x %d x %d, %d pairs, form %d\n", need, bytes, batch, la, lb, pairs, form);
                failures++;
              }
            }
}

// Planning under a limit on the address space: an error, not an exception
// through the C interface.
static void memory() {
  const Layout many({1 << 20, 4, 1}, {1, 1, 1});
  const dm::Side t = many.side();
  struct rlimit lim;
  getrlimit(RLIMIT_AS, &lim);
  const struct rlimit before = lim;
  FILE *f = fopen("/proc/self/statm", "r");
  long pages = 0;
  if (f == nullptr || fscanf(f, "%ld", &pages) != 1) failures++;
  if (f != nullptr) fclose(f);
  lim.rlim_cur = (rlim_t)pages * sysconf(_SC_PAGESIZE) + (4 << 20);  // 4 MiB more than now
  setrlimit(RLIMIT_AS, &lim);
  {
    dm::TableBuilder tb;
    dm::PendingPass pp;
    // 2^20 lines of 4 points: 16 MiB of line bases
    if (dm::plan_pass(many.comm, t, t, 1, 1, false, nullptr, nullptr, tb, &pp) || !dm::error_pending()) {
      printf("a pass was planned within 4 MiB, or without an error\n");
      failures++;
    }
    dm::PendingBlock pb;
    if (dm::plan_block(t, t, {1}, 1, false, nullptr, nullptr, tb, &pb, 1)) {
      printf("a block pass was planned within 4 MiB\n");
      failures++;
    }
  }
  setrlimit(RLIMIT_AS, &before);
}

// Every line length within a tile: a schedule of its stages that fits the
// launch arguments and multiplies to the length.
static void stages() {
  for (int n = 1; n <= dm::fft_tile_capacity(0, 1); n++) {
    std::vector<int> rad;
    long long m = 1;
    const bool ok = dm::choose_radices(n, &rad, true);
    for (int r : rad) m *= r;
    if (!ok || m != n || (int)rad.size() > dm::kMaxStages) {
      printf("length %d: %zu stages\n", n, rad.size());
      failures++;
    }
  }
}

// Workgroups of passes over few lines: as many as tiles hold the lines where
// the whole array is less than 20 KiB; more from there on, and where a
// direct-sum stage has work for them.
static void few_lines() {
  const struct {
    int n, lines;
    bool whole[2];  // complex float, complex double
  } at[] = {{32, 39, {true, true}},    {32, 40, {true, false}}, {32, 79, {true, false}},  {32, 80, {false, false}},
            {3, 100, {true, true}},    {104, 8, {true, true}},  {8, 104, {true, true}},   {600, 4, {true, true}},
            {256, 16, {false, false}}, {79, 15, {false, false}}, {106, 38, {false, false}}};
  for (const auto &c : at)
    for (int t : {0, 1})
      for (int dbl : {0, 1}) {
        const Layout l(t == 0 ? std::vector<int>{c.n, c.lines} : std::vector<int>{c.lines, c.n}, {1, 1});
        const dm::Side s = l.side();
        dm::TableBuilder tb;
        dm::PendingPass pp;
        const int most = dm::fft_tile_capacity(dbl, t == 0) / c.n, held = (c.lines + most - 1) / most;
        if (!dm::plan_pass(l.comm, s, s, t, dbl, false, nullptr, nullptr, tb, &pp) || (pp.L.tiles_u == held) != c.whole[dbl]) {
          printf("%d lines of %d along axis %d, dbl %d: %lld tiles, %d hold them\n", c.lines, c.n, t, dbl,
                 (long long)pp.L.tiles_u, held);
          failures++;
        }
      }
}

int main(int argc, char **argv) {
  dm_set_error_mode(1);
  const std::string check = argc > 1 ? argv[1] : "";
  if (check == "lds") lds();
  else if (check == "tables") tables();
  else if (check == "reshape") reshape();
  else if (check == "memory") memory();
  else if (check == "stages") stages();
  else if (check == "few_lines") few_lines();
  else return 2;
  if (failures == 0) printf("OK\n");
  return failures != 0;
}
