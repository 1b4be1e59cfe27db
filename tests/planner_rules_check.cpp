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
#define main planner_check_main
#include "planner_check.cpp"
#undef main

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
