// planner_rules_check.cpp -- host-only checks of the batch planner's rules (CPU
// test, no GPU): what planner_check.cpp builds, with commands of its own.
//
// stdin, one command per line (x decimal, key=value options first: shape=TxK,
// alpha=<factor>, c=<wheel>, any of which makes the context a tuned one; budget=
// bytes of a batch's state):
//   groups x x ...   "groups <size> <size> ..." of the plan, by increasing x
//   needs x x ...    "needs <R> <P> <Y>": the tables the batch asks for, which must
//                    reach the end of its last P2 segment in the context's shape
//   bytes x x ...    "bytes <state> <estimate>": what the batch's plan takes and what
//                    a batch-mode server admits it by (tables=1: P2 by lookups)
//   claim left grid  "claim <tiles>": main tiles a streaming block claims at once
//   check x x ...    "check <tiles>": check_plan's conditions, and that the wheel-stage
//                    descriptors cover their odd m, every partial sum has one
//                    descriptor, and the carry descriptors name their rows
#define main planner_check_main
#include "planner_check.cpp"
#undef main
#include "../cudapix_amd/csrc/cpx_stream.hpp"

struct Cmd {
  std::string what;
  std::vector<HostQuery> hq;
};

static void plan_into(cpx_ctx *c, Cmd &cmd, Plan &pl, uint32_t p2mode = 0)
{
  choose_p2tab(c, cmd.hq, TERM_ALL, p2mode);
  uint64_t R = 0, P = 0, Y = 0;
  for (const HostQuery &h : cmd.hq) plan_needs(c, h, TERM_ALL, c->shape.seg_bits(), &R, &P, &Y);
  fake_tables(c, R, P, Y);
  CHECK(build_plan(c, cmd.hq, TERM_ALL, pl) == CPX_OK, "build_plan");
}

static void check_descriptors(const cpx_ctx *c, const Plan &pl, const Caps &k)
{
  for (size_t i = 0; i < pl.q.size(); i++) {
    const QueryDev &d = pl.q[i];
    const QPlan &qp = pl.qps[i];
    std::vector<int> used(qp.parts, 0);
    for (const std::vector<BlockDesc> *v : {&qp.ord, &qp.triv, &qp.easy, &qp.fin, &qp.dir, &qp.p2d})
      for (const BlockDesc &b : *v) {
        CHECK(b.query == i && b.part < qp.parts, "descriptor's query and part");
        used[b.part]++;
      }
    for (int n : used) CHECK(n == 1, "one descriptor a partial sum");
    if (d.small) continue;
    CHECK(d.c <= d.cs && d.cs + d.nstage <= c->nprimes, "stages inside the prime list");
    const uint32_t h0 = d.n_ord_parts + d.n_triv_parts + d.n_easy_parts, h1 = h0 + d.n_hard_parts;
    if (d.cs > d.c) {
      uint64_t at = d.y / c->h_primes[d.cs - 1] / 2;      // odd m = 2i + 1 from here
      for (const BlockDesc &b : qp.dir) {
        CHECK(b.part >= h0 && b.part < h1, "wheel stages among the hard parts");
        CHECK(b.begin == at && b.end > b.begin, "wheel-stage ranges adjoin");
        at = b.end;
      }
      CHECK(at == (d.y + 1) / 2, "wheel stages to y");
    } else {
      CHECK(qp.dir.empty(), "no wheel stages");
    }
    uint64_t st = 0;
    for (const BlockDesc &b : qp.fin) {
      const uint64_t s0 = (uint32_t)b.begin;
      CHECK(b.part >= h0 && b.part < h1, "carry among the hard parts");
      CHECK(s0 == st && b.end > s0 && b.end - s0 <= CPX_FIN_STAGES, "carry stages adjoin");
      st = b.end;
      uint64_t rows = 0;
      while (rows < d.hard_nseg && qp.rowinfo[rows].act > s0) rows++;
      CHECK(b.begin >> 32 == rows, "rows of a carry descriptor");
    }
    CHECK(st == d.nstage, "carry of every stage");
    for (uint64_t s = d.p2_seg0; s < d.p2_seg0 + d.p2_nseg; s++)
      CHECK(d.mrow_base + qp.rowinfo[s].mrow + qp.rowinfo[s].nrep <= k.mrows, "P2 outputs of every replica");
  }
}

int main()
{
  std::string line;
  while (std::getline(std::cin, line)) {
    if (line.empty()) continue;
    static std::vector<uint32_t> primes;      // (kept from line to line: the longest list)
    static uint64_t limit = 0;
    cpx_ctx ctx;
    cpx_ctx *c = &ctx;
    c->h_primes.swap(primes);
    c->nprimes = c->h_primes.size();
    c->prime_limit = limit;
    c->opts.c = 6;
    c->opts.alpha = 0;
    c->opts.fresh_tables = 0;
    c->shape = {512, 32};
    std::istringstream in(line);
    Cmd cmd;
    bool tables = false;
    in >> cmd.what;
    if (cmd.what == "claim") {
      uint64_t left;
      uint32_t grid;
      in >> left >> grid;
      std::printf("claim %llu\n", (unsigned long long)cpx_main_claim_run(left, grid));
      primes.swap(c->h_primes);
      continue;
    }
    std::string tok;
    while (in >> tok) {
      const size_t eq = tok.find('=');
      if (eq != std::string::npos) {
        const std::string k = tok.substr(0, eq), v = tok.substr(eq + 1);
        if (k == "tables") { tables = v == "1"; continue; }
        if (k == "budget") { c->state_budget = (uint64_t)parse_u128(v); continue; }
        if (k == "shape") CHECK(std::sscanf(v.c_str(), "%dx%d", &c->shape.threads, &c->shape.kwords) == 2, "shape");
        if (k == "alpha") c->alpha_scale = std::atof(v.c_str());
        if (k == "c") c->opts.c = (uint32_t)std::atoi(v.c_str());
        c->shape_tuned = true;
        continue;
      }
      HostQuery h;
      CHECK(make_host_query(c, parse_u128(tok), 0, 0, &h) == CPX_OK, "make_host_query");
      cmd.hq.push_back(h);
    }
    if (cmd.what == "groups") {
      Plan pl;
      plan_into(c, cmd, pl);
      std::printf("groups");
      for (const GroupDev &g : pl.groups) std::printf(" %u", g.n);
      std::printf("\n");
    } else if (cmd.what == "check") {
      if (tables) fake_tables(c, cmd.hq[0].zt, cmd.hq[0].sqrtx, cmd.hq[0].y);
      const ShapeScope scope(c, cmd.hq);
      Plan pl;
      plan_into(c, cmd, pl);
      Caps k{};
      grown_caps(Caps{}, needed_caps(pl), k);
      const Layout L = make_layout(k);
      std::vector<char> image(L.plan_bytes);
      pack_plan(L, pl, image.data());
      check_plan(c, pl, L, k, false);
      check_descriptors(c, pl, k);
      std::printf("check %zu\n", pl.tiles.size());
    } else if (cmd.what == "bytes") {
      uint64_t sum = 0, top = 0;
      for (size_t i = 0; i < cmd.hq.size(); i++) {
        sum += plan_bytes_estimate(c, cmd.hq[i]);
        if (cmd.hq[i].x > cmd.hq[top].x) top = i;
      }
      const uint64_t est = batch_bytes_estimate(c, sum, cmd.hq.size(), cmd.hq[top]);
      if (tables) fake_tables(c, cmd.hq[top].zt, cmd.hq[top].sqrtx, cmd.hq[top].y);
      const ShapeScope scope(c, cmd.hq);
      Plan pl;
      plan_into(c, cmd, pl, 1);
      const Layout L = make_layout(needed_caps(pl));
      std::printf("bytes %zu %llu\n", L.plan_bytes + L.out_bytes, (unsigned long long)est);
    } else if (cmd.what == "needs") {
      choose_p2tab(c, cmd.hq, TERM_ALL, 1);
      uint64_t R, P, Y;
      const ShapeScope scope(c, cmd.hq);
      batch_needs(c, cmd.hq, TERM_ALL, &R, &P, &Y);
      for (const HostQuery &h : cmd.hq) {
        const uint64_t SI = c->shape.seg_ints();
        if (!h.small && h.y < h.sqrtx) CHECK(P >= cpx_isqrt128((u128)(h.zt / SI + 1) * SI), "primes of the last segment");
      }
      std::printf("needs %llu %llu %llu\n", (unsigned long long)R, (unsigned long long)P, (unsigned long long)Y);
    } else {
      CHECK(false, "unknown command");
    }
    primes.swap(c->h_primes);
    limit = c->prime_limit;
  }
  return 0;
}
