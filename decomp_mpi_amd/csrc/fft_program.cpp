// Pass programs: tile axes, walk modes, radix schedules and device tables.
#include "fft_program.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <numeric>

#include "logger.h"

namespace dm {

Side make_side(const HostLayout &h, i64 slot) {
  Side s;
  s.h = h;
  s.slot = slot;
  s.abs.resize(h.ndim);
  s.order.resize(h.ndim);
  for (int d = 0; d < h.ndim; d++) {
    s.abs[d].resize(h.L[d]);
    for (int g = 0; g < h.L[d]; g++) s.abs[d][g] = (i64)h.rank_part[d][g] * slot + h.m[d] * h.off[d][g];
    s.order[d].resize(h.L[d]);
    std::iota(s.order[d].begin(), s.order[d].end(), 0);
    const auto &a = s.abs[d];
    std::stable_sort(s.order[d].begin(), s.order[d].end(), [&](int x, int y) { return a[x] < a[y]; });
  }
  return s;
}

// Odd prime factors one stage each; powers of two in radix-8 stages with one
// 16/4/2 stage for the remainder.  any_prime: primes above 13 become stages
// of the direct-sum kernel, last in the schedule (the pass kernel's
// general-radix stage); without it such a length is refused.
bool choose_radices(int n, std::vector<int> *out, bool any_prime) {
  out->clear();
  if (n < 1) return false;
  std::vector<int> odd, big;
  const int primes[] = {13, 11, 7, 5, 3};
  for (int p : primes)
    while (n % p == 0) {
      odd.push_back(p);
      n /= p;
    }
  int k = 0;
  while (n % 2 == 0) {
    n /= 2;
    k++;
  }
  if (any_prime)
    for (int p = 17; n > 1 && p <= n; p += 2)
      while (n % p == 0) {
        big.push_back(p);
        n /= p;
      }
  if (n != 1) return false;
  std::vector<int> pw;
  while (k >= 3) {
    pw.push_back(8);
    k -= 3;
  }
  if (k == 1) {
    if (!pw.empty()) pw.back() = 16;
    else pw.push_back(2);
  } else if (k == 2) {
    pw.push_back(4);
  }
  out->insert(out->end(), pw.begin(), pw.end());
  out->insert(out->end(), odd.begin(), odd.end());
  out->insert(out->end(), big.begin(), big.end());
  return true;
}

std::vector<double> roots(int n) {
  std::vector<double> w(2 * (size_t)n);
  const long double tau = 6.283185307179586476925286766559005768L;
  const long double h = 0.70710678118654752440084436210484903L;
  const long double tc[8] = {1, h, 0, -h, -1, -h, 0, h};
  const long double ts[8] = {0, h, 1, h, 0, -h, -1, -h};
  for (int k = 0; k < n; k++) {
    long double c, s;
    if ((8LL * k) % n == 0) {  // multiples of pi/4 exactly
      c = tc[8LL * k / n];
      s = ts[8LL * k / n];
    } else {
      long double a = tau * (long double)k / (long double)n;
      c = cosl(a);
      s = sinl(a);
    }
    w[2 * (size_t)k] = (double)c;
    w[2 * (size_t)k + 1] = (double)(-s);
  }
  return w;
}

void twiddle_image(const double *w, size_t n, int dbl, void *dst) {
  if (dbl) {
    memcpy(dst, w, n * 2 * sizeof(double));
    return;
  }
  // bfloat16 of x: the high half of its float bits, rounded to nearest even
  auto bf16 = [](double x) -> uint32_t {
    float f = (float)x;
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
  };
  uint32_t *e = (uint32_t *)dst;
  for (size_t i = 0; i < n; i++) {
    const double re = w[2 * i], im = w[2 * i + 1];
    const float hr = (float)re, hi = (float)im;
    memcpy(&e[4 * i], &hr, 4);
    memcpy(&e[4 * i + 1], &hi, 4);
    e[4 * i + 2] = bf16(re - (double)hr) | (bf16(im - (double)hi) << 16);
    e[4 * i + 3] = 0;
  }
}

bool axis_supported(int n, int dbl, std::string *why) {
  char msg[160];
  std::vector<int> rad;
  const int cap = fft_tile_capacity(dbl, 1);
  if (n > cap) {
    snprintf(msg, sizeof msg, "axis length %d exceeds the %d-point tile of the %s pass", n, cap,
             dbl ? "complex-double" : "complex-float");
  } else if (!choose_radices(n, &rad, true) || (int)rad.size() > kMaxStages) {
    snprintf(msg, sizeof msg, "axis length %d takes more than %d stages", n, kMaxStages);
  } else {
    return true;
  }
  if (why) *why = msg;
  return false;
}

size_t TableBuilder::space(size_t bytes) {
  const size_t at = host.n, need = at + ((bytes + 255) & ~(size_t)255);
  if (need > host.cap) {
    const size_t cap = std::max(need, host.cap + host.cap / 2);
    char *p = (char *)realloc(host.p, cap);
    if (p == nullptr) throw std::bad_alloc();
    host.p = p;
    host.cap = cap;
  }
  memset(host.p + at + bytes, 0, need - at - bytes);
  host.n = need;
  return at;
}

size_t TableBuilder::put(const void *src, size_t bytes) {
  const size_t at = space(bytes);
  memcpy(host.p + at, src, bytes);
  return at;
}

static bool is_identity(const std::vector<int> &o) {
  for (size_t i = 0; i < o.size(); i++)
    if (o[i] != (int)i) return false;
  return true;
}

static bool plan_pass_tables(dm_comm_t comm, const Side &I, const Side &U, int t, int dbl, bool inverse,
                             const void *in, void *out, TableBuilder &tb, PendingPass *pp, int ctw) {
  int nd = I.h.ndim;
  FftLaunch &L = pp->L;
  memset(&L, 0, sizeof L);
  L.ndim = nd;
  for (int d = 0; d < nd; d++) L.L[d] = I.h.L[d];
  L.t = t;
  L.N = I.h.L[t];
  int cap = fft_tile_capacity(dbl, 1);
  if (L.N > cap) {
    raise_error(comm, "FFT: axis %d of length %d exceeds the %d-point pass tile", t, L.N, cap);
    return false;
  }
  std::vector<int> rad;
  if (!choose_radices(L.N, &rad, true) || (int)rad.size() > kMaxStages) {
    raise_error(comm, "FFT: axis length %d takes more than %d stages", L.N, kMaxStages);
    return false;
  }
  L.nstage = (int)rad.size();
  for (int s = 0; s < L.nstage; s++) L.radix[s] = rad[s];
  auto fastest_other = [&](const Side &s) {
    int best = -1;
    for (int d = 0; d < nd; d++) {
      if (d == t || s.h.L[d] <= 1) continue;
      if (best < 0 || s.h.m[d] < s.h.m[best] || (s.h.m[d] == s.h.m[best] && d > best)) best = d;
    }
    return best;
  };
  bool in_row = (I.h.fastest == t) || fastest_other(I) < 0;
  bool out_row = (U.h.fastest == t) || fastest_other(U) < 0;
  int u = out_row ? fastest_other(I) : fastest_other(U);
  L.u = u;
  L.in_row = in_row ? 1 : 0;
  L.out_row = out_row ? 1 : 0;
  // rank positions along t of a side whose ranks have strides of their own
  auto positions = [&](const Side &s) {
    std::vector<int> v;
    if (!s.h.uniform) {
      v = s.h.rank_part[t];
      std::sort(v.begin(), v.end());
      v.erase(std::unique(v.begin(), v.end()), v.end());
    }
    return v;
  };
  const std::vector<int> pos_in = positions(I), pos_out = positions(U);
  L.sin.uniform = I.h.uniform ? 1 : 0;
  L.sin.np = (int)pos_in.size();
  L.sin.form = L.sin.np > kLinePositions ? 2 : 0;
  L.sout.uniform = U.h.uniform ? 1 : 0;
  L.sout.np = (int)pos_out.size();
  L.sout.form = L.sout.np > kLinePositions ? 2 : 0;
  L.dbl = dbl;
  L.ctw = (!dbl && ctw) ? 1 : 0;
  const int np_most = std::max(std::max(L.sin.np, L.sout.np), 1);
  // positions per line of the sides that keep their lines' bases in LDS
  const int np_lds = std::max(std::max(L.sin.form == 2 ? 1 : L.sin.np, L.sout.form == 2 ? 1 : L.sout.np), 1);
  // Small arrays: lines per tile are halved while a pass has fewer than 192
  // tiles for the 256 CUs and its rows are longer than 64 bytes (so 5 complex
  // doubles become 3; stopping at 64 bytes exactly, 8 lines for 6, a forward
  // of 68x8x24 complex floats took 43.5 us for 40.5).  What is left to win
  // there is the latency of one tile, which falls with its points per thread
  // (64^3 complex double over pencils 22.0 -> 20.1 us a transform, 61x21x100
  // on 12 ranks 182 -> 104, 75x200 on 6 62 -> 43).  At 256 tiles
  // 2940x576 lost (145 -> 153 us: rows of half the width for nothing, all
  // CUs were busy); at 512 and 1024 arrays of a million points did (71 -> 87
  // and 105 us for 256x208x72).  Less than 20 KiB of points stay in one tile:
  // more workgroups only fetch the code more often.  Forwards spread and
  // whole: 84x14 complex floats 35.7 and 33.7 us, 78x20 34.9 and 32.5, 65x35
  // 38.7 and 37.5; beyond, 96x30 36.8 and 38.0, 27x125 38.7 and 40.7; complex
  // doubles 90x12 28.1 and 28.3, 105x15 36.7 and 39.3, 45x45 38.4 and 42.6.
  // A direct-sum stage has work for more workgroups (45x79 complex floats
  // 52 and 109).
  long long lines = 1;
  for (int d = 0; d < nd; d++)
    if (d != t) lines *= I.h.L[d];
  auto spread = [&](int T) {
    const int least = 64 / (dbl ? 16 : 8);
    if (lines * L.N * (dbl ? 16 : 8) < (20 << 10) && std::all_of(rad.begin(), rad.end(), has_radix_kernel)) return T;
    while (T > least && lines / T < 192) T = (T + 1) / 2;
    return T;
  };
  if (u >= 0) {
    // column walk at a line stride of 64 KiB or more: wide rows pay for the
    // lower occupancy of the wide tile -- for lines of 256 points or more
    // (the phase order's 16- and 32-point sub-axis passes ran slower in it:
    // FFT_2 6.15 -> 5.54 ms per 512^3 step without)
    const size_t es = dbl ? 16 : 8;
    bool wide = L.N >= 256 && ((!in_row && (size_t)I.h.m[t] * es >= (64u << 10)) ||
                               (!out_row && (size_t)U.h.m[t] * es >= (64u << 10)));
    static const bool nowide = getenv("DM_NO_WIDE") != nullptr;
    auto height = [&](bool w) {
      const int T = spread(std::max(1, std::min(std::min(fft_tile_capacity(dbl, !(in_row && out_row), w) / L.N, I.h.L[u]), 512)));
      // per-line address data of a non-uniform side: 16 KiB of LDS at most
      return np_lds > 1 ? std::max(1, std::min(T, kLineEntries / np_lds)) : T;
    };
    L.T = height(wide && !nowide);
    // the wide tile (136 KiB and up to 16 of twiddles) leaves no room for the
    // line data of many positions; the other tiles do: at most 118 KiB in all
    if (fft_lds_bytes(L) > kLdsBytes) L.T = height(false);
    L.tiles_u = (I.h.L[u] + L.T - 1) / L.T;
  } else {
    L.T = 1;
    L.tiles_u = 1;
  }
  // Non-temporal data accesses measured faster on every pass (512^3: up to
  // 10%) except the stores of a pass whose output is a column walk at a line
  // stride of 64 KiB or more: there the hint on the loads alone is best
  // (complex float: 2.58 -> 2.50 ms per 512^3 step against the hint on both).
  {
    // (complex double: no hint at all there, 4.63 ms against 4.85 with the
    // hint on its loads)
    const size_t es = dbl ? 16 : 8;
    static const bool nont = getenv("DM_NO_NONTEMPORAL") != nullptr;
    const bool far = !out_row && (size_t)U.h.m[t] * es >= (64u << 10);
    L.stream_in = (nont || (far && dbl)) ? 0 : 1;
    L.stream_out = (nont || far) ? 0 : 1;
  }
  L.nbatch = 0;
  for (int d = 0; d < nd; d++)
    if (d != t && d != u) L.batch_axis[L.nbatch++] = d;
  // A row walk on both sides whose u axis holds less than half a tile of
  // lines: each tile takes all L[u] lines for k consecutive values of the
  // fastest batch axis (k dividing its length), so tiles stay full (the
  // sub-axis passes of the phase order: 16- or 32-point lines, 16 or 32 of
  // them along u).
  L.merge_v = -1;
  L.merge_k = 1;
  if (u >= 0 && L.nbatch > 0 && in_row && out_row) {
    // (the most that leave 192 tiles; fewer tiles than that whatever k is:
    // the height of small arrays)
    const int lu = I.h.L[u], v = L.batch_axis[L.nbatch - 1];
    const int full = std::min(fft_tile_capacity(dbl, 0) / L.N, 512), low = spread(full);
    if (np_most == 1)
      for (int k = full / lu; k >= 2; k--)
        if (I.h.L[v] % k == 0 && (lines / (lu * k) >= 192 || lu * k <= low)) {
          L.merge_v = v;
          L.merge_k = k;
          L.T = lu * k;
          L.tiles_u = 1;
          break;
        }
  }
  const long long ntiles = fft_pass_tiles(L);
  long long batch = 1;
  for (int k = 0; k < L.nbatch; k++) batch *= I.h.L[L.batch_axis[k]];
  if (ntiles >= (1LL << 31)) {
    raise_error(comm, "FFT: %lld workgroups exceed the launch limit", ntiles);
    return false;
  }
  L.inverse = inverse ? 1 : 0;
  // per-axis tables one after another
  for (int d = 1; d < nd; d++) L.at[d] = L.at[d - 1] + L.L[d - 1];
  auto joined = [&](const auto &tab) {
    std::decay_t<decltype(tab[0])> v;
    for (int d = 0; d < nd; d++) v.insert(v.end(), tab[d].begin(), tab[d].end());
    return tb.put(v.data(), v.size() * sizeof(v[0]));
  };
  pp->in_off = joined(I.abs);
  pp->out_off = joined(U.abs);
  // rank-dependent strides: owner, local offset and per-rank stride tables
  auto side = [&](const Side &s, FftSide &fs, PendingSide &ps, const std::vector<int> &pos) {
    fs.proc_used = s.h.proc_used;
    fs.slot = s.slot;
    // offsets along t affine (x * m_t: axis t local to every rank, in
    // order), or in runs of R = 2^k points at a jump J per run (axis t in
    // equal blocks over the ranks: (x >> k) * J + (x & (R - 1)) * m_t)
    fs.aff = 0;
    fs.jump = 0;
    if (s.h.uniform && s.h.m[t] > 0) {
      bool affine = true;
      for (int x = 0; x < s.h.L[t] && affine; x++) affine = s.h.rank_part[t][x] == 0 && s.h.off[t][x] == x;
      static const bool noaff = getenv("DM_NO_AFFINE") != nullptr;
      if (affine && !noaff) fs.aff = s.h.m[t];
      const std::vector<i64> &a = s.abs[t];
      const i64 m = s.h.m[t];
      const int n = s.h.L[t];
      if (!affine && !noaff && a[0] == 0) {
        int R = 1;
        while (R < n && a[R] == a[R - 1] + m) R++;
        if (R < n && (R & (R - 1)) == 0) {
          int k = 0;
          while ((1 << k) < R) k++;
          const i64 J = a[R];
          bool ok = J != 0;
          for (int x = 0; x < n && ok; x++) ok = a[x] == (i64)(x >> k) * J + (i64)(x & (R - 1)) * m;
          if (ok) {
            fs.jump = J;
            fs.rstride = m;
            fs.rsh = k;
            fs.rmask = R - 1;
          }
        }
      }
    }
    if (s.h.uniform) return;
    std::vector<int> xt(2 * (size_t)L.N);
    bool in_order = fs.np == 1;
    for (int x = 0; x < L.N; x++) {
      xt[2 * (size_t)x] = (int)(std::lower_bound(pos.begin(), pos.end(), s.h.rank_part[t][x]) - pos.begin());
      xt[2 * (size_t)x + 1] = s.h.off[t][x];
      in_order = in_order && s.h.off[t][x] == x;
    }
    if (in_order) fs.form = 1;
    ps.xt = tb.put(xt.data(), xt.size() * sizeof(int));
    ps.posrank = tb.put(pos.data(), pos.size() * sizeof(int));
    ps.rank = joined(s.h.rank_part);
    ps.off = joined(s.h.off);
    ps.strides = tb.put(s.h.strides.data(), s.h.strides.size() * sizeof(i64));
  };
  side(I, L.sin, pp->sin, pos_in);
  side(U, L.sout, pp->sout, pos_out);
  if (in_row && !is_identity(I.order[t])) pp->ord_in = (long)tb.put(I.order[t].data(), L.N * sizeof(int));
  if (out_row && !is_identity(U.order[t])) pp->ord_out = (long)tb.put(U.order[t].data(), L.N * sizeof(int));
  if (u >= 0) {
    // tile lines follow the address order of the column-walked side
    const Side &cs = out_row ? I : U;
    if (!is_identity(cs.order[u])) pp->ord_u = (long)tb.put(cs.order[u].data(), I.h.L[u] * sizeof(int));
  }
  // Per-tile line bases for uniform sides: one coalesced load per tile in
  // the kernel instead of a chain of lookups (bounded to 64 MiB of tables).
  // Non-uniform sides form theirs in the kernel (90 x 126 x 100 on 6 ranks:
  // 86 us against 81 with tables, but 371 against 566 for a first pass).
  {
    const long long nlines = (long long)L.tiles_u * batch * L.T;
    if (L.merge_k == 1 && I.h.uniform && U.h.uniform && nlines * 16 <= (64LL << 20)) {
      const std::vector<int> *ou = nullptr;
      if (pp->ord_u >= 0) ou = &((out_row ? I : U).order[u]);
      // u coordinate of every line of a row of tiles
      const int nu = L.tiles_u * L.T;
      std::vector<int> cu(nu, 0), g(nd, 0);
      for (int l = 0; l < nu && u >= 0; l++)
        if (l < I.h.L[u]) cu[l] = ou ? (*ou)[l] : l;
      auto fill = [&](const Side &s) {
        const size_t where = tb.space(nlines * sizeof(i64));
        std::vector<i64> au(nu, 0);
        for (int l = 0; l < nu && u >= 0; l++) au[l] = s.abs[u][cu[l]];
        std::fill(g.begin(), g.end(), 0);
        i64 *at = (i64 *)(tb.host.data() + where);
        for (long long b = 0; b < batch; b++) {
          i64 base = 0;
          for (int k = 0; k < L.nbatch; k++) base += s.abs[L.batch_axis[k]][g[L.batch_axis[k]]];
          for (int l = 0; l < nu; l++) at[l] = base + au[l];
          at += nu;
          for (int k = L.nbatch - 1; k >= 0; k--) {  // the next batch coordinate
            const int d = L.batch_axis[k];
            if (++g[d] < I.h.L[d]) break;
            g[d] = 0;
          }
        }
        return (long)where;
      };
      pp->line_in = fill(I);
      pp->line_out = fill(U);
    }
  }
  // Twiddles in stage order: stage s (Ns = product of the earlier radices,
  // radix R) holds w^(jj * r * N / (Ns * R)) for r = 1..R-1, jj < Ns at
  // index (Ns - 1) + (r - 1) * Ns + jj, so the lanes of a wave (consecutive
  // jj) read consecutive entries.  The stages telescope to N - 1 entries.
  const std::vector<double> &root = tb.root->of(L.N);
  std::vector<double> w(2 * (size_t)L.N, 0.0);
  {
    int ns = 1;
    for (int st = 0; st < L.nstage; st++) {
      int R = L.radix[st];
      int stride = L.N / (ns * R);
      for (int r = 1; r < R; r++)
        for (int jj = 0; jj < ns; jj++) {
          size_t at = (size_t)(ns - 1) + (size_t)(r - 1) * ns + jj;
          size_t k = (size_t)jj * r * stride;
          w[2 * at] = root[2 * k];
          w[2 * at + 1] = root[2 * k + 1];
        }
      ns *= R;
    }
    // after the N stage entries: w_p^m = w^(m N / p), m < p, for each stage
    // of a radix without a kernel of its own, in stage order
    for (int st = 0; st < L.nstage; st++) {
      int R = L.radix[st];
      if (has_radix_kernel(R)) continue;
      for (int m = 0; m < R; m++) {
        size_t k = (size_t)m * (L.N / R);
        w.push_back(root[2 * k]);
        w.push_back(root[2 * k + 1]);
      }
    }
  }
  const size_t ntw = w.size() / 2;
  std::vector<char> img(ntw * 16);
  twiddle_image(w.data(), ntw, dbl, img.data());
  pp->tw = (long)tb.put(img.data(), img.size());
  L.in = in;
  L.out = out;
  auto form = [](const FftSide &f) {
    if (f.aff) return std::string(" affine");
    if (f.jump) return " affine in runs of " + std::to_string(f.rmask + 1);
    return std::string("");
  };
  logger(comm, "FFT pass: axis %d (N %d, %d stages) lines along %d, T %d, %lld workgroups, in %s stride %lld%s, out %s stride %lld%s%s%s\n",
         t, L.N, L.nstage, u, L.T, ntiles, in_row ? "row" : "column", (long long)I.h.m[t],
         form(L.sin).c_str(), out_row ? "row" : "column", (long long)U.h.m[t], form(L.sout).c_str(),
         L.stream_in ? ", non-temporal loads" : "", L.stream_out ? ", non-temporal stores" : "");
  return true;
}

bool plan_pass(dm_comm_t comm, const Side &I, const Side &U, int t, int dbl, bool inverse, const void *in,
               void *out, TableBuilder &tb, PendingPass *pp, int ctw) {
  try {
    return plan_pass_tables(comm, I, U, t, dbl, inverse, in, out, tb, pp, ctw);
  } catch (const std::bad_alloc &) {  // the callers are C entry points
    raise_error(comm, "FFT: no host memory for the tables of the pass over axis %d", t);
    return false;
  }
}

// Radices of a block pass stage by stage: powers of two in 16s, 8s and 4s
// (a 16-point axis is one butterfly of a thread's 16 points).
static bool block_radices(int n, std::vector<int> *out) {
  out->clear();
  for (int p : {7, 5, 3})
    while (n % p == 0) {
      out->push_back(p);
      n /= p;
    }
  int k = 0;
  while (n % 2 == 0) {
    n /= 2;
    k++;
  }
  if (n != 1) return false;
  // 2^k with as few stages as 16 allows, even ones: 2^5 = 8 4, 2^6 = 8 8
  const int stages = (k + 3) / 4;
  for (int i = 0; i < stages; i++) {
    const int b = (k + (stages - i) - 1) / (stages - i);
    out->push_back(1 << b);
    k -= b;
  }
  return true;
}

// Fastest axis of a layout outside `axes` (smallest stride among the axes
// longer than one), or -1.
static int fastest_outside(const Side &s, const std::vector<int> &axes) {
  int best = -1;
  for (int d = 0; d < s.h.ndim; d++) {
    if (s.h.L[d] <= 1 || std::find(axes.begin(), axes.end(), d) != axes.end()) continue;
    if (best < 0 || s.h.m[d] < s.h.m[best]) best = d;
  }
  return best;
}

// The line axis of a block pass (the fastest axis outside its axes) and
// lines per tile: as many as fit, but where the contiguous axis is among the
// transformed ones (whole rows anyway) no more than leave a tile for each of
// the 256 CUs (75 x 45 x 45 complex floats: 19 full tiles 84 us a step, 75
// of one plane 67).
static int block_lines(const Side &I, const std::vector<int> &axes, int dbl, int *T) {
  long long points = 1, total = 1;
  for (int d : axes) points *= I.h.L[d];
  for (int l : I.h.L) total *= l;
  const int u = fastest_outside(I, axes);
  *T = 1;
  if (u < 0) return u;
  const int lu = I.h.L[u];
  int t = (int)std::max(1LL, std::min<long long>(fft_block_capacity(dbl) / points, lu));
  if (std::find(axes.begin(), axes.end(), I.h.fastest) != axes.end()) {
    const long long batch = total / points / lu;
    while (t > 1 && batch * ((lu + t - 1) / t) < 256) t = (t + 1) / 2;
  }
  *T = t;
  return u;
}

bool block_fits(const Side &I, const Side &U, const std::vector<int> &axes, int dbl) {
  if (!I.h.uniform || !U.h.uniform || axes.empty() || axes.size() > DM_BLOCK_DIMS - 1) return false;
  long long points = 1, total = 1;
  size_t stages = 0;
  std::vector<int> rad;
  for (int d : axes) {
    points *= I.h.L[d];
    if (points > fft_block_capacity(dbl) || !block_radices(I.h.L[d], &rad)) return false;
    stages += rad.size();
  }
  for (int l : I.h.L) total *= l;
  if (stages > kBlockStages) return false;
  int T;
  const int u = block_lines(I, axes, dbl, &T);
  // both sides in runs of 128 bytes along the same axis, or the whole array
  // in a tile
  const int es = dbl ? 16 : 8;
  if (U.h.fastest != I.h.fastest && points * T < total) return false;
  for (const Side *s : {&I, &U}) {
    const int f = s->h.fastest;
    const int run = std::find(axes.begin(), axes.end(), f) != axes.end() ? I.h.L[f] : (f == u ? T : 1);
    if (run * es < 128 && points * T < total) return false;
  }
  return total / points * 16 <= (64LL << 20);  // the line bases
}

static bool plan_block_tables(const Side &I, const Side &U, const std::vector<int> &axes, int dbl, bool inverse,
                              const void *in, void *out, TableBuilder &tb, PendingBlock *pb, int ctw, int wq) {
  FftBlock &B = pb->B;
  memset(&B, 0, sizeof B);
  const int nd = I.h.ndim;
  int T;
  const int u = block_lines(I, axes, dbl, &T);
  auto magic = [](int d) { return magic_for(d); };
  // the tile's dimensions, innermost first: by the input's strides
  std::vector<int> dims = axes;
  if (u >= 0) dims.push_back(u);
  std::stable_sort(dims.begin(), dims.end(), [&](int x, int y) { return I.h.m[x] < I.h.m[y]; });
  B.ndim = (int)dims.size();
  B.line_dim = -1;
  B.points = 1;
  std::vector<int> stride(nd, 0);
  std::vector<i64> oi, oo;
  for (int k = 0; k < B.ndim; k++) {
    const int d = dims[k], n = d == u ? T : I.h.L[d];
    if (d == u) B.line_dim = k;
    B.dim[k].n = n;
    B.dim[k].m_n = magic(n);
    B.dim[k].at = (int)oi.size();
    stride[d] = B.points;
    B.points *= n;
    for (int x = 0; x < n; x++) {
      oi.push_back(d == u ? 0 : I.abs[d][x]);
      oo.push_back(d == u ? 0 : U.abs[d][x]);
    }
  }
  if (u < 0) {  // one line: its base in an entry (and a dimension) of its own
    B.line_dim = B.ndim;
    B.dim[B.ndim].n = 1;
    B.dim[B.ndim].m_n = magic(1);
    B.dim[B.ndim].at = (int)oi.size();
    B.ndim++;
    oi.push_back(0);
    oo.push_back(0);
  }
  B.ntab = (int)oi.size();
  pb->off_in = tb.put(oi.data(), oi.size() * sizeof(i64));
  pb->off_out = tb.put(oo.data(), oo.size() * sizeof(i64));
  // stages: the outermost transformed axis first and last (fused with the
  // load and the store when its radices are powers of two), the others
  // between, innermost last
  std::vector<int> by_stride = axes;
  std::stable_sort(by_stride.begin(), by_stride.end(), [&](int x, int y) { return stride[x] > stride[y]; });
  std::vector<double> tw;
  std::vector<std::vector<BlockStage>> of(by_stride.size());
  for (size_t a = 0; a < by_stride.size(); a++) {
    const int d = by_stride[a], n = I.h.L[d];
    std::vector<int> rad;
    block_radices(n, &rad);
    if (a == 0 && rad.size() > 1 && (rad[0] & (rad[0] - 1)) != 0) std::reverse(rad.begin(), rad.end());
    const std::vector<double> &root = tb.root->of(n);
    int ns = 1;
    for (int r : rad) {
      BlockStage st{};
      st.dim = (int)(std::find(dims.begin(), dims.end(), d) - dims.begin());
      st.radix = r;
      st.s = stride[d];
      st.span = stride[d] * n;
      st.nr = n / r;
      st.ns = ns;
      st.m_s = magic(st.s);
      st.m_nr = magic(st.nr);
      st.m_ns = magic(st.ns);
      st.tw = (int)(tw.size() / 2);
      for (int q = 1; q < r && ns > 1; q++)
        for (int jj = 0; jj < ns; jj++) {
          const size_t k = (size_t)jj * q * (n / (ns * r));
          tw.push_back(root[2 * k]);
          tw.push_back(root[2 * k + 1]);
        }
      of[a].push_back(st);
      ns *= r;
    }
  }
  std::vector<BlockStage> seq;
  const bool split = of[0].size() > 1;
  for (size_t i = 0; i < of[0].size(); i++)
    if (!split || i + 1 < of[0].size()) seq.push_back(of[0][i]);
  for (size_t a = by_stride.size(); a-- > 1;)  // innermost first: the next outer axis may end the pass
    for (auto &st : of[a]) seq.push_back(st);
  if (split) seq.push_back(of[0].back());
  B.nstage = (int)seq.size();
  for (int i = 0; i < B.nstage; i++) B.st[i] = seq[i];
  auto pow2 = [](int r) { return (r & (r - 1)) == 0; };
  // (along the contiguous dimension a butterfly's points are nr apart: with
  // fewer than 8 butterflies a line, lanes would be whole rows apart)
  B.fuse_in = pow2(seq[0].radix) && (seq[0].s > 1 || seq[0].nr >= 8);
  B.fuse_out = B.nstage >= 2 && pow2(seq.back().radix) && (seq.back().s > 1 || seq.back().nr >= 8);
  if (tw.empty()) tw.assign(2, 0.0);
  B.ntw = (int)(tw.size() / 2);
  std::vector<char> img(tw.size() / 2 * 16);
  twiddle_image(tw.data(), tw.size() / 2, dbl, img.data());
  pb->tw = tb.put(img.data(), img.size());
  // line bases
  std::vector<int> batch;
  long long nbatch = 1;
  for (int d = 0; d < nd; d++)
    if (d != u && std::find(axes.begin(), axes.end(), d) == axes.end()) {
      batch.push_back(d);
      nbatch *= I.h.L[d];
    }
  // slowest first, so that neighbouring tiles are close in memory
  std::stable_sort(batch.begin(), batch.end(), [&](int x, int y) { return I.h.m[x] > I.h.m[y]; });
  B.lines = u < 0 ? 1 : I.h.L[u];
  B.tiles_u = (B.lines + T - 1) / T;
  B.tiles = nbatch * B.tiles_u;
  const int nu = B.tiles_u * T;
  auto fill = [&](const Side &s) {
    const size_t where = tb.space((size_t)nbatch * nu * sizeof(i64));
    i64 *to = (i64 *)(tb.host.data() + where);
    std::vector<int> g(nd, 0);
    std::vector<i64> along(nu, 0);
    for (int l = 0; l < nu && u >= 0; l++) along[l] = s.abs[u][l < B.lines ? I.order[u][l] : 0];
    for (long long b = 0; b < nbatch; b++) {
      i64 base = 0;
      for (int d : batch) base += s.abs[d][g[d]];
      for (int l = 0; l < nu; l++) to[b * nu + l] = base + along[l];
      for (size_t k = batch.size(); k-- > 0;) {
        if (++g[batch[k]] < s.h.L[batch[k]]) break;
        g[batch[k]] = 0;
      }
    }
    return where;
  };
  pb->base_in = fill(I);
  pb->base_out = fill(U);
  if (wq >= 0) {
    const auto at = std::find(batch.begin(), batch.end(), wq);
    if (at == batch.end() || !B.fuse_in || axes.size() != 1) return false;
    B.wn = I.h.L[axes[0]];
    B.wlen = I.h.L[wq];
    B.wdiv = 1;
    for (auto k = at + 1; k != batch.end(); ++k) B.wdiv *= I.h.L[*k];
    const int N = B.wn * B.wlen;
    const std::vector<double> &w = tb.root->of(N);
    std::vector<char> wi((size_t)N * 16);
    twiddle_image(w.data(), N, dbl, wi.data());
    pb->wtab = (long)tb.put(wi.data(), wi.size());
  }
  static const bool nont = getenv("DM_NO_NONTEMPORAL") != nullptr;
  B.stream_in = B.stream_out = nont ? 0 : 1;
  B.inverse = inverse ? 1 : 0;
  B.dbl = dbl;
  B.ctw = !dbl && ctw ? 1 : 0;
  B.in = in;
  B.out = out;
  fft_block_lds(&B);
  return B.lds <= 160 * 1024 && B.tiles < (1LL << 31);
}

bool plan_block(const Side &I, const Side &U, const std::vector<int> &axes, int dbl, bool inverse, const void *in,
                void *out, TableBuilder &tb, PendingBlock *pb, int ctw, int wq) {
  try {
    return plan_block_tables(I, U, axes, dbl, inverse, in, out, tb, pb, ctw, wq);
  } catch (const std::bad_alloc &) {
    return false;
  }
}

void *finalize_passes(dm_comm_t comm, TableBuilder &tb, std::vector<PendingPass> &pp,
                      std::vector<FftLaunch> *out, std::vector<PendingBlock> *pb, std::vector<FftBlock> *blocks) {
  void *mem = device_alloc(std::max<size_t>(tb.host.size(), 256));
  if (mem == nullptr) {
    raise_error(comm, "FFT: device allocation of %zu bytes of tables failed", tb.host.size());
    return nullptr;
  }
  if (!tb.host.empty()) h2d(mem, tb.host.data(), tb.host.size());
  char *b = (char *)mem;
  out->clear();
  if (pb != nullptr) {
    blocks->clear();
    for (auto &p : *pb) {
      FftBlock B = p.B;
      B.off_in = (const i64 *)(b + p.off_in);
      B.off_out = (const i64 *)(b + p.off_out);
      B.base_in = (const i64 *)(b + p.base_in);
      B.base_out = (const i64 *)(b + p.base_out);
      B.twiddle = b + p.tw;
      B.wtab = p.wtab >= 0 ? b + p.wtab : nullptr;
      blocks->push_back(B);
    }
  }
  for (auto &p : pp) {
    FftLaunch L = p.L;
    if (L.block) {
      out->push_back(L);
      continue;
    }
    L.off_in = (const i64 *)(b + p.in_off);
    L.off_out = (const i64 *)(b + p.out_off);
    auto side = [&](FftSide &fs, const PendingSide &ps) {
      if (fs.uniform) return;
      fs.rank = (const int *)(b + ps.rank);
      fs.off = (const int *)(b + ps.off);
      fs.strides = (const i64 *)(b + ps.strides);
      fs.xt = (const int *)(b + ps.xt);
      fs.posrank = (const int *)(b + ps.posrank);
    };
    side(L.sin, p.sin);
    side(L.sout, p.sout);
    L.ord_in = p.ord_in >= 0 ? (const int *)(b + p.ord_in) : nullptr;
    L.ord_out = p.ord_out >= 0 ? (const int *)(b + p.ord_out) : nullptr;
    L.ord_u = p.ord_u >= 0 ? (const int *)(b + p.ord_u) : nullptr;
    L.line_in_tab = p.line_in >= 0 ? (const i64 *)(b + p.line_in) : nullptr;
    L.line_out_tab = p.line_out >= 0 ? (const i64 *)(b + p.line_out) : nullptr;
    L.twiddle = b + p.tw;
    out->push_back(L);
  }
  return mem;
}

bool layout_usable(dm_comm_t comm, const char *what, const HostLayout &h, size_t region_elems) {
  if (!h.offsets_ok) {
    raise_error(comm, "FFT: the %s decomposition has a negative offset or stride", what);
    return false;
  }
  for (int d = 0; d < h.ndim; d++)
    for (int g = 0; g < h.L[d]; g++)
      if (h.rank_part[d][g] >= DM_NO_OWNER) {
        raise_error(comm, "FFT: coordinate %d of axis %d of the %s decomposition has no owner", g, d, what);
        return false;
      }
  for (int r = 0; r < h.proc_used; r++)
    if ((size_t)h.slot_extent[r] > region_elems) {
      raise_error(comm, "FFT: rank %d needs %lld elements of %s, the buffer region holds %zu", r,
                  (long long)h.slot_extent[r], what, region_elems);
      return false;
    }
  return true;
}

}  // namespace dm

namespace dm {

// Axis d of h as two sub-axes over g = y + A_d * z: sub-axis 2d is y (A_d
// points), sub-axis 2d+1 is z (L_d / A_d points).  The owner and the local
// offset must be sums of a y part and a z part (the split FFT's A and B
// decompositions are: Interleave(Block(A, ga), B) gives rank(y) and
// z + B * off(y); BlockWithFactor(A * B, A, gb) gives rank(z) and
// y + A * (z % (bs / A))).  Each part's offsets are divided by their common
// step, which goes into the sub-axis' memory stride.
bool split_layout(const HostLayout &h, const std::vector<int> &A, HostLayout *out, std::string *why) {
  const int nd = h.ndim;
  if (2 * nd > DM_MAX_DIMS) {
    *why = "too many axes to split";
    return false;
  }
  HostLayout s;
  s.ndim = 2 * nd;
  s.proc_used = h.proc_used;
  s.L.assign(2 * nd, 1);
  s.rank_part.assign(2 * nd, std::vector<int>());
  s.off.assign(2 * nd, std::vector<int>());
  s.strides.assign((size_t)h.proc_used * 2 * nd, 0);
  s.uniform = h.uniform;
  s.slot_extent = h.slot_extent;
  s.offsets_ok = h.offsets_ok;
  for (int d = 0; d < nd; d++) {
    const int L = h.L[d], a = A[d];
    if (a < 1 || L % a != 0) {
      *why = "factor does not divide the axis";
      return false;
    }
    const int b = L / a;
    const auto &rp = h.rank_part[d];
    const auto &of = h.off[d];
    std::vector<int> ry(a), rz(b), oy(a), oz(b);
    for (int z = 0; z < b; z++) {
      rz[z] = rp[a * z];
      oz[z] = of[a * z];
    }
    for (int y = 0; y < a; y++) {
      ry[y] = rp[y] - rp[0];
      oy[y] = of[y] - of[0];
    }
    for (int z = 0; z < b; z++)
      for (int y = 0; y < a; y++) {
        const int g = y + a * z;
        if (rp[g] >= DM_NO_OWNER || rp[g] != ry[y] + rz[z] || of[g] != oy[y] + oz[z]) {
          *why = "the decomposition is not separable along the split";
          return false;
        }
      }
    auto step_of = [](const std::vector<int> &o) {
      int st = 0;
      for (int v : o) st = std::gcd(st, v < 0 ? -v : v);
      return st > 0 ? st : 1;
    };
    const int sy = step_of(oy), sz = step_of(oz);
    for (auto &v : oy) v /= sy;
    for (auto &v : oz) v /= sz;
    s.L[2 * d] = a;
    s.L[2 * d + 1] = b;
    s.rank_part[2 * d] = ry;
    s.rank_part[2 * d + 1] = rz;
    s.off[2 * d] = oy;
    s.off[2 * d + 1] = oz;
    for (int r = 0; r < h.proc_used; r++) {
      const i64 m = h.strides[(size_t)r * nd + d];
      s.strides[(size_t)r * 2 * nd + 2 * d] = m * sy;
      s.strides[(size_t)r * 2 * nd + 2 * d + 1] = m * sz;
    }
  }
  s.m.assign(s.strides.begin(), s.strides.begin() + 2 * nd);
  // fastest sub-axis: smallest stride among those longer than one; ties ->
  // the later sub-axis
  int best = 2 * nd - 1;
  i64 bs = -1;
  for (int i = 2 * nd - 1; i >= 0; i--) {
    if (s.L[i] <= 1) continue;
    if (bs < 0 || s.m[i] < bs) {
      bs = s.m[i];
      best = i;
    }
  }
  s.fastest = best;
  *out = s;
  return true;
}

}  // namespace dm
