// san_host.cpp -- CPU test program of the library's host code under the address
// and undefined-behaviour sanitizers (test infrastructure: built by
// `make -C fidibench_amd/csrc sanitize` with the host side of every source
// instrumented, run by tests/test_host_sanitize.py; never shipped).
//
// It calls every entry point whose work is host logic -- the checkpoint
// schedule, the reference's checksum/std folds, the maps of the device's
// parallel form of them, the two VTK writers, the
// raw-file header checks on good, truncated, foreign and malformed files,
// the CLI parser, argument validation of the handle/tape/filter
// constructors (which stop before any device work) and the tuning-variable
// parser -- on small and edge-case inputs.  A sanitizer report aborts the
// run; a wrong result exits 1.
//
//   san_host            the checks above
//   san_host tuning     the same process with malformed tuning variables set
//   san_host rows       ... with a shape for the FP64 rows kernel set
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/fidibench_amd/CmdLineArgs.hpp"
#include "../../include/fidibench_amd/fdb_filter.h"
#include "../../include/fidibench_amd/fdb_upwind.h"
#include "fdb_fold_map.h"
#include "fdb_internal.h"

namespace {

int g_fail = 0;

void check(bool ok, const char* what) {
  if (!ok) {
    std::fprintf(stderr, "FAILED: %s (%s)\n", what, fdb_last_error());
    ++g_fail;
  }
}

std::string tmp(const char* name) {
  const char* d = std::getenv("TMPDIR");
  return std::string(d && *d ? d : "/tmp") + "/fdb_san_" + name;
}

void plans() {
  // Every (steps, snapshots) pair on a small grid, caps below the plan
  // length (the output is cut, the count still returned) and T = 400.
  for (int T = 0; T <= 40; T += (T < 10 ? 1 : 7)) {
    for (int s = 0; s <= 6; ++s) {
      int64_t fw = -1;
      const int n = fdb_ckpt_plan(T, s, nullptr, nullptr, 0, &fw);
      check(n >= 0 && fw >= 0, "ckpt_plan length");
      std::vector<int> a(n + 1), b(n + 1);
      check(fdb_ckpt_plan(T, s, a.data(), b.data(), n, &fw) == n, "ckpt_plan fill");
      check(fdb_ckpt_plan(T, s, a.data(), b.data(), n / 2, &fw) == n, "ckpt_plan cut");
    }
  }
  for (int s : {1, 2, 3, 5, 165}) {
    int64_t fw = 0;
    const int n = fdb_ckpt_plan(400, s, nullptr, nullptr, 0, &fw);
    std::vector<int> a(n), b(n);
    check(fdb_ckpt_plan(400, s, a.data(), b.data(), n, &fw) == n && fw > 0, "ckpt_plan 400");
  }
  check(fdb_ckpt_plan(-1, 0, nullptr, nullptr, 0, nullptr) == FDB_ERR_INVALID, "plan T < 0");
  check(fdb_ckpt_plan(5, -1, nullptr, nullptr, 0, nullptr) == FDB_ERR_INVALID, "plan s < 0");
}

void folds_and_vtk() {
  const double f[7] = {1.0, -0.0, 1e-310, 3.5, -2.25, 1e300, -1e300};
  check(fdb_host_checksum(f, 7) == ((((((1.0 + -0.0) + 1e-310) + 3.5) + -2.25) + 1e300) + -1e300),
        "left fold");
  check(fdb_host_checksum(f, 0) == 0.0, "empty fold");
  (void)fdb_host_std(f, 4);
  const uint64_t n3[3] = {3, 4, 5}, n2[2] = {4, 6}, n1[1] = {7};
  const double len[3] = {1.0, 1.5, 2.0}, xmin[3] = {0, 0, 0};
  std::vector<double> g(60);
  for (size_t i = 0; i < g.size(); ++i) g[i] = 0.1 * (double)i - 2.0;
  check(fdb_host_save_vtk(3, n3, len, g.data(), tmp("a.vtk").c_str()) == FDB_OK, "save_vtk 3d");
  check(fdb_host_save_vtk(2, n2, len, g.data(), tmp("b.vtk").c_str()) == FDB_OK, "save_vtk 2d");
  check(fdb_host_save_vtk(1, n1, len, g.data(), tmp("c.vtk").c_str()) == FDB_OK, "save_vtk 1d");
  check(fdb_host_save_vtk(4, n3, len, g.data(), tmp("d.vtk").c_str()) == FDB_ERR_INVALID,
        "save_vtk ndims");
  check(fdb_host_save_vtk(1, n1, len, g.data(), "/nonexistent_dir/x.vtk") == FDB_ERR_IO,
        "save_vtk io");
  check(fdb_host_write_vtk(3, n3, xmin, len, g.data(), "f", tmp("e.vtk").c_str()) == FDB_OK,
        "write_vtk 3d");
  check(fdb_host_write_vtk(1, n1, xmin, len, g.data(), "f", tmp("f.vtk").c_str()) == FDB_OK,
        "write_vtk 1d");
}

// One value at a time and in runs of 8, 64 and 512 joined pairwise, as the
// fold kernel's lanes, waves and blocks join them; then the host's step.
// Values: multiples of a quarter unit and both neighbours of each (ties and
// what lies next to a tie on either side), of both signs, added to even and
// odd significands of both signs in several binades.
void fold_maps() {
  uint64_t r = 88172645463325252ull;
  auto rnd = [&] { return r ^= r << 13, r ^= r >> 7, r ^= r << 17; };
  auto value = [&](double u) {
    double q = (double)(int64_t)(rnd() % 17) - 8.0;
    q *= 0.25 * u;
    const uint64_t side = rnd() % 3;
    return side == 0 ? q : std::nextafter(q, side == 1 ? -1e300 : 1e300);
  };
  int bad = 0;
  for (int ex : {-900, -3, 0, 1, 52, 53, 700})
    for (int neg = 0; neg < 2; ++neg)
      for (int rep = 0; rep < 400; ++rep) {
        const double u = std::ldexp(1.0, ex - 52);
        const int n = rep < 200 ? 1 : 512;
        std::vector<double> x(n);
        for (double& v : x) v = value(u);
        const uint64_t m = (3ull << 51) + rnd() % 4;
        const double s0 = (neg ? -1.0 : 1.0) * std::ldexp((double)m, ex - 52);
        double want = s0;
        for (double v : x) want = want + v;
        std::vector<fdb::FoldMap> runs;
        for (int i = 0; i < n; i += 8) {
          fdb::FoldMap f = fdb::fold_identity();
          for (int k = i; k < std::min(n, i + 8); ++k)
            fdb::fold_append(f, std::ldexp(neg ? -x[k] : x[k], 52 - ex));
          runs.push_back(f);
        }
        while (runs.size() > 1) {
          for (size_t i = 0; 2 * i < runs.size(); ++i)
            runs[i] = fdb::fold_then(runs[2 * i], runs[2 * i + 1]);
          runs.resize(runs.size() / 2);
        }
        const fdb::FoldMap& f = runs[0];
        double got = s0;
        const fdb::FoldRec rec{f.d0, f.d1, f.lo, f.hi, ex, neg, fdb::kFoldMapped, -1};
        const bool applies = fdb::fold_step(rec, nullptr, (uint64_t)n, (uint64_t)n, &got);
        if ((!applies || got != want) && ++bad <= 4)
          std::fprintf(stderr, "fold map: n %d ex %d s0 %a x0 %a want %a got %a\n", n, ex, s0, x[0],
                       want, got);
      }
  check(bad == 0, "fold maps equal the sequential loop");
}

// The chunks of a field of equal values, mapped where the guessed sum (in
// another order) lets them: every map must apply to the loop's own sum, which
// drifts from the guess as all additions round alike.  Values that bring the
// sum to a power of two at a chunk's start, and next to them.
void fold_guesses() {
  const uint64_t chunk = 2048, n = 600 * chunk;
  int bad = 0, mapped = 0;
  for (uint64_t at : {3, 77, 300, 599})
    for (int near = -40; near <= 40; ++near) {
      double x = std::ldexp(1.0, 3) / (double)(at * chunk);
      for (int i = 0; i < std::abs(near); ++i) x = std::nextafter(x, near < 0 ? 0.0 : 1.0);
      double s = 0.0;
      for (uint64_t c = 0; c * chunk < n; ++c) {
        const double guess = (double)(c * chunk) * x;
        const int ex = std::ilogb(guess);
        double want = s;
        for (uint64_t i = 0; i < chunk; ++i) want = want + x;
        if (guess > 0.0) {
          fdb::FoldMap m = fdb::fold_identity();
          fdb::fold_append(m, std::ldexp(x, 52 - ex));
          for (uint64_t k = 1; k < chunk; k *= 2) m = fdb::fold_then(m, m);
          if (fdb::fold_fits(std::ldexp(guess, 52 - ex), m.lo, m.hi, fdb::fold_slack(n))) {
            const fdb::FoldRec rec{m.d0, m.d1, m.lo, m.hi, ex, 0, fdb::kFoldMapped, -1};
            double got = s;
            ++mapped;
            if ((!fdb::fold_step(rec, nullptr, chunk, chunk, &got) || got != want) && ++bad <= 4)
              std::fprintf(stderr, "fold guess: at %d near %d chunk %d s %a guess %a\n", (int)at,
                           near, (int)c, s, guess);
          }
        }
        s = want;
      }
    }
  check(bad == 0 && mapped > 4 * 81 * 500, "guessed sums hold");
}

// The fold's plan: every chunk of fields up to 16 MB can be copied out, and
// what larger ones copy fits the 64 MiB staging buffer.
void fold_plans() {
  for (uint64_t n : {65536ull, 65537ull, 400000ull, 2097152ull, 2097153ull, 1ull << 27, 1ull << 33}) {
    const fdb::FoldPlan p = fdb::fold_plan(n);
    check(p.nchunks * p.chunk >= n && (p.nchunks - 1) * p.chunk < n && p.nchunks <= 16384, "chunks");
    check(n * 8 > (16u << 20) || p.slots == p.nchunks, "every chunk has a slot");
    check(p.slots >= 8 && p.slots <= p.nchunks && p.host_bytes <= (64u << 20) &&
              p.host_bytes >= p.gather_off + p.slots * p.chunk * 8 && p.dev_bytes > p.host_bytes,
          "slots");
  }
}

void write_file(const std::string& path, const std::vector<unsigned char>& bytes) {
  FILE* fp = std::fopen(path.c_str(), "wb");
  if (!fp) {
    check(false, "write temp file");
    return;
  }
  if (!bytes.empty()) std::fwrite(bytes.data(), 1, bytes.size(), fp);
  std::fclose(fp);
}

std::vector<unsigned char> raw(uint32_t nd, uint32_t dt, uint64_t a, uint64_t b, uint64_t c,
                               size_t payload) {
  std::vector<unsigned char> v(64 + payload, 0);
  std::memcpy(v.data(), "FDBFLD01", 8);
  std::memcpy(v.data() + 8, &nd, 4);
  std::memcpy(v.data() + 12, &dt, 4);
  const uint64_t n[3] = {a, b, c};
  std::memcpy(v.data() + 16, n, 24);
  return v;
}

void raw_headers() {
  const std::string p = tmp("f.raw");
  int nd = 0, dt = 0;
  uint64_t n[3] = {0, 0, 0}, st = 0, sd = 0;
  write_file(p, raw(3, 0, 4, 5, 6, 4 * 5 * 6 * 8));
  check(fdb_host_raw_info(p.c_str(), &nd, &dt, n, &st, &sd) == FDB_OK && nd == 3 && n[2] == 6,
        "raw good");
  check(fdb_host_raw_info(p.c_str(), nullptr, nullptr, nullptr, nullptr, nullptr) == FDB_OK,
        "raw good, no outputs");
  write_file(p, raw(3, 0, 4, 5, 6, 4 * 5 * 6 * 8 - 1));
  check(fdb_host_raw_info(p.c_str(), &nd, &dt, n, &st, &sd) == FDB_ERR_IO, "raw truncated");
  write_file(p, raw(2, 1, 1u << 31, 1u << 31, 1, 0));
  check(fdb_host_raw_info(p.c_str(), &nd, &dt, n, &st, &sd) == FDB_ERR_IO, "raw huge");
  write_file(p, raw(3, 0, ~0ull, ~0ull, ~0ull, 0));
  check(fdb_host_raw_info(p.c_str(), &nd, &dt, n, &st, &sd) == FDB_ERR_IO, "raw overflow");
  write_file(p, raw(9, 0, 1, 1, 1, 8));
  check(fdb_host_raw_info(p.c_str(), &nd, &dt, n, &st, &sd) == FDB_ERR_IO, "raw ndims");
  write_file(p, raw(1, 77, 1, 1, 1, 8));
  check(fdb_host_raw_info(p.c_str(), &nd, &dt, n, &st, &sd) == FDB_ERR_IO, "raw dtype");
  write_file(p, std::vector<unsigned char>(10, 'x'));
  check(fdb_host_raw_info(p.c_str(), &nd, &dt, n, &st, &sd) == FDB_ERR_IO, "raw foreign");
  write_file(p, {});
  check(fdb_host_raw_info(p.c_str(), &nd, &dt, n, &st, &sd) == FDB_ERR_IO, "raw empty");
  check(fdb_host_raw_info(tmp("none.raw").c_str(), &nd, &dt, n, &st, &sd) == FDB_ERR_IO,
        "raw missing");
  check(fdb_host_raw_info(nullptr, &nd, &dt, n, &st, &sd) == FDB_ERR_INVALID, "raw null");
}

void cli() {
  const std::vector<std::vector<std::string>> cases = {
      {}, {"-numCells", "16", "-numSteps", "3", "-std"}, {"32", "10"},
      {"-numCells"}, {"-numSteps", "5", "-numCells", "24", "-numCells", "20"},
      {"-std", "-std", "-vtk"}, {"-bogus"}, {"-h"}, {"-precision", "bf16", "-timeBlock", "8"},
      {"-numCells", "-3"}, {"-numCells", "99999999999999999999"}};
  for (const auto& c : cases) {
    std::vector<std::string> keep = {"upwindCxx"};
    keep.insert(keep.end(), c.begin(), c.end());
    std::vector<char*> argv;
    for (auto& s : keep) argv.push_back(&s[0]);
    argv.push_back(nullptr);
    fidibench::CmdLineArgs a;
    a.set("-numCells", 128, "Number of cells along each axis.");
    a.set("-numSteps", 10, "Number of time steps.");
    a.set("-vtk", false, "Write VTK files.");
    a.set("-std", false, "Print the standard deviation.");
    a.set("-precision", "f64", "Storage type.");
    a.set("-timeBlock", 1, "Steps per pass.");
    a.set("-dt", 0.5, "Time step.");
    if (a.parse((int)keep.size(), argv.data())) {
      (void)a.get<int>("-numCells");
      (void)a.get<int>("-nope");
      (void)a.get<double>("-dt");
      (void)a.get<std::string>("-precision");
      (void)a.get<bool>("-std");
    }
  }
}

void constructors() {
  const double v[3] = {0.3, -0.2, 0.1}, len[3] = {1, 1, 1};
  const uint64_t ok[3] = {8, 8, 8}, zero[3] = {8, 0, 8};
  const uint64_t wraps[3] = {1ull << 21, 1ull << 21, 1ull << 20};  // 2^62 cells
  fdb_upwind_t* h = nullptr;
  check(fdb_upwind_create(0, v, len, ok, FDB_F64, &h) == FDB_ERR_INVALID, "create ndims");
  check(fdb_upwind_create(3, v, len, zero, FDB_F64, &h) == FDB_ERR_INVALID, "create zero");
  check(fdb_upwind_create(3, v, len, ok, 9, &h) == FDB_ERR_INVALID, "create dtype");
  check(fdb_upwind_create(3, nullptr, len, ok, FDB_F64, &h) == FDB_ERR_INVALID, "create null");
  check(fdb_upwind_create(3, v, len, wraps, FDB_F64, &h) == FDB_ERR_INVALID, "create bytes");
  check(fdb_upwind_create(3, v, len, ok, FDB_F64, nullptr) == FDB_ERR_INVALID, "create out");
  check(fdb_upwind_advect(nullptr, 1, 0.1) == FDB_ERR_INVALID, "advect null");
  check(fdb_upwind_destroy(nullptr) == FDB_OK, "destroy null");
  fdb_tape_t* t = nullptr;
  check(fdb_tape_create(3, ok, v, len, 0.01, 0, FDB_F64, FDB_F64, 1 << 20, &t) ==
            FDB_ERR_INVALID, "tape steps");
  check(fdb_tape_create(3, wraps, v, len, 0.01, 4, FDB_F64, FDB_F64, 1 << 20, &t) ==
            FDB_ERR_INVALID, "tape bytes");
  check(fdb_tape_create(3, ok, v, len, 0.01, 4, FDB_F64, FDB_BF16_SR, 1 << 20, &t) ==
            FDB_ERR_INVALID, "tape lam dtype");
  check(fdb_tape_set_method(nullptr, FDB_GRAD_SHIFT) == FDB_ERR_INVALID, "tape method null");
  fdb_filter_t* f = nullptr;
  const int offs[6] = {0, 0, 1, 0, 9, 0};
  const double w[3] = {1.0, 0.5, 0.25};
  const uint64_t d2[2] = {16, 16};
  check(fdb_filter_create(2, d2, len, len, 3, offs, w, &f) == FDB_ERR_INVALID, "filter offset");
  check(fdb_filter_create(2, d2, len, len, 0, offs, w, &f) == FDB_ERR_INVALID, "filter terms");
  const uint64_t big[3] = {(1ull << 31) - 1, (1ull << 31) - 1, 1};
  check(fdb_filter_create(3, big, len, len, 1, offs, w, &f) == FDB_ERR_INVALID, "filter bytes");
  // Valid arguments get as far as the device: none here.
  const int rc = fdb_upwind_create(3, v, len, ok, FDB_F64, &h);
  check(rc == FDB_ERR_NODEV || (rc == FDB_OK && fdb_upwind_destroy(h) == FDB_OK), "create nodev");
}

// Which one-step launches over a 2-D field the plane kernel makes; rows_64:
// FDB_ROWS_CFG_8 is set.
void one_step_routes(bool rows_64) {
  const uint64_t n[3] = {40, 50, 60};
  const double v[3] = {0.3, -0.2, 0.1}, len[3] = {1, 1, 1};
  fdb::Grid3 g2, g3;
  check(fdb::make_grid(2, n, v, len, 1e-3, &g2) && fdb::make_grid(3, n, v, len, 1e-3, &g3), "grid");
  check(fdb::one_step_by_plane(FDB_F64, g2) == !rows_64, "2-D FP64 step");
  check(fdb::one_step_by_plane(FDB_F32, g2), "2-D FP32 step");
  check(!fdb::one_step_by_plane(FDB_BF16, g2) && !fdb::one_step_by_plane(FDB_BF16_SR, g2),
        "2-D bf16 step");
  check(!fdb::one_step_by_plane(FDB_F64, g3), "3-D step");
}

// Rows of a k-step launch's blocks.
int picked_rows(int dtype, uint64_t n0, uint64_t n1, uint64_t n2, int k) {
  const uint64_t n[3] = {n0, n1, n2};
  const double v[3] = {0.3, -0.2, 0.1}, len[3] = {1, 1, 1};
  fdb::Grid3 g;
  check(fdb::make_grid(3, n, v, len, 1e-3, &g), "grid");
  int rows = 0;
  check(fdb::picked_chunk(dtype, g, k, &rows) > 0, "a pick");
  return rows;
}

void picked_shapes() {
  check(picked_rows(FDB_BF16, 256, 256, 256, 6) == 64, "bf16 6 steps: two blocks per CU");
  check(picked_rows(FDB_F64, 158, 102, 177, 2) == 36, "FP64 2 steps: tall waves");
  check(picked_rows(FDB_F32, 13, 1794, 12, 2) == 36, "FP32 2 steps: tall waves");
  check(picked_rows(FDB_F64, 16, 16, 16, 4) == 16, "FP64 4 steps: short waves");
  check(picked_rows(FDB_F64, 3088, 19, 404, 8) == 56, "FP64 8 steps: two planes a trip");
}

// The tiles of fused passes over long grids fill the device: 8 tiles an axis-0
// chunk, one block per CU, where 1 to 24 chunks leave a quarter of it idle.
void long_grid_chunks() {
  const uint64_t n[3] = {3088, 19, 404};
  const double v[3] = {0.3, -0.2, 0.1}, len[3] = {1, 1, 1};
  fdb::Grid3 g;
  check(fdb::make_grid(3, n, v, len, 1e-3, &g), "grid");
  int rows = 0;
  const int64_t chunk = fdb::picked_chunk(FDB_F64, g, 7, &rows);
  check(chunk > 0 && rows > 7, "a pick");
  const int64_t tiles = (404 + 56) / 57 * ((19 + rows - 8) / (rows - 7));
  const int64_t blocks = tiles * ((3088 + chunk - 1) / chunk);
  check(blocks % 256 == 0 || blocks % 256 > 224, "blocks fill the last round");
  // Every grid gets a chunk within its planes.
  for (uint64_t n0 : {1, 2, 23, 24, 25, 600, 601, 5000, 1000000})
    for (int dt : {FDB_F64, FDB_F32, FDB_BF16})
      for (int k : {2, 3, 4, 6, 7, 8}) {
        const uint64_t m[3] = {n0, 3, 5};
        check(fdb::make_grid(3, m, v, len, 1e-3, &g), "grid");
        const int64_t c = fdb::picked_chunk(dt, g, k, nullptr);
        check(c >= 1 && c <= (int64_t)n0, "chunk within the planes");
      }
}

// Grids of up to four rows a plane take blocks of two waves, of two rows each.
void one_step_shapes() {
  const double v[3] = {0.3, -0.2, 0.1}, len[3] = {1, 1, 1};
  for (int dt : {FDB_F64, FDB_F32, FDB_BF16, FDB_BF16_SR})
    for (uint64_t n1 : {1, 2, 4, 5, 40}) {
      const uint64_t n[3] = {7, n1, 900};
      fdb::Grid3 g, g1;
      check(fdb::make_grid(3, n, v, len, 1e-3, &g), "grid");
      check(fdb::one_step_waves(dt, g) == (n1 <= 4 ? 2 : 4), "waves of a step");
      check(fdb::make_grid(1, n + 2, v, len, 1e-3, &g1), "grid");
      check(fdb::one_step_waves(dt, g1) == 2, "waves of a 1-D step");
    }
}

// Star stencils over planes of eight rows: the block form where the grid is
// small or narrow, the marching kernel otherwise.
void filter_routes() {
  auto block = [](int64_t n0, int64_t n1, int64_t n2, int R) {
    fdb::FilterGeom g{};
    g.n[0] = n0, g.n[1] = n1, g.n[2] = n2;
    const int order[5] = {0, 1, 2, 1, 0}, lo[5] = {-R, -R, -R, 1, 1}, hi[5] = {-1, -1, R, R, R};
    for (int b = 0; b < 5; ++b)
      for (int k = lo[b]; k <= hi[b]; ++k) g.off[g.nt++][order[b]] = k;
    fdb::FilterPlan p{};
    check(fdb::plan_filter(g, &p) == hipSuccess, "filter plan");
    return p.block;
  };
  check(!block(20000, 8, 6, 2) && !block(128, 8, 2000, 2) && !block(2000, 8, 64, 2), "marching");
  check(block(20000, 8, 6, 1) && block(1000, 8, 64, 2) && block(30, 8, 30000, 2) &&
            block(4000, 9, 150, 2) && block(100, 8, 7, 2), "blocks");
}

}  // namespace

int main(int argc, char** argv) {
  if (argc > 1 && std::strcmp(argv[1], "tuning") == 0) {
    // Malformed tuning variables: every launching constructor refuses
    // with FDB_ERR_INVALID, naming the variable.
    setenv("FDB_TB_CFG_8_6", "9,8,0,1,2,3,4,5,6,7,8,9", 1);
    setenv("FDB_ROWS_CFG", "8,2", 1);
    const double v[3] = {0.3, -0.2, 0.1}, len[3] = {1, 1, 1};
    const uint64_t ok[3] = {8, 8, 8};
    fdb_upwind_t* h = nullptr;
    check(fdb_upwind_create(3, v, len, ok, FDB_F64, &h) == FDB_ERR_INVALID &&
              std::strstr(fdb_last_error(), "FDB_") != nullptr, "tuning refused");
    fdb_tape_t* t = nullptr;
    check(fdb_tape_create(3, ok, v, len, 0.01, 4, FDB_F64, FDB_F64, 1 << 30, &t) ==
              FDB_ERR_INVALID, "tuning refused (tape)");
  } else if (argc > 1 && std::strcmp(argv[1], "rows") == 0) {
    setenv("FDB_ROWS_CFG_8", "4,2,0,1", 1);
    one_step_routes(true);
  } else {
    one_step_routes(false);
    long_grid_chunks();
    picked_shapes();
    one_step_shapes();
    filter_routes();
    plans();
    folds_and_vtk();
    fold_maps();
    fold_guesses();
    fold_plans();
    raw_headers();
    cli();
    constructors();
  }
  if (g_fail) {
    std::fprintf(stderr, "%d check(s) failed\n", g_fail);
    return 1;
  }
  std::printf("san_host ok%s%s\n", argc > 1 ? " " : "", argc > 1 ? argv[1] : "");
  return 0;
}
