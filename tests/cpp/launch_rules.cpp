// Prints what the library's launch rules choose, host arithmetic only: one line per line of input.
//   insert key=value ...        choose_fr_insert of a launch: "<which> <blocks> <threads> <lds> <kernel>"
//   batch_tuner key=value ...   what the batch tuner times: "<kernel>,<boxFixed>" of the first schedule
//                               and of the candidates over it, then the number of schedules
//   op_tuner key=value ...      the kernels of an operation's schedule candidates
//   op_key key=value ...        the key of an operation's tuning result: Init told of `init` spaces
//   batch_key key=value ...     ... of a batch of one job
//   core key=value ...          cells of a volume's core and bricks beside it (exact launches)
//   depth key=value ...         the depth scale of a batch's launch and of a plain operation's
#include <dlfcn.h>

#include <cstdio>
#include <iostream>
#include <map>
#include <sstream>
#include <string>

#include "../../umpalumpa_amd/csrc/fr_host.hpp"
#include "../../umpalumpa_amd/csrc/launch.hpp"

namespace {

std::map<std::string, double> g_args;
double arg(const char *key, double otherwise = 0)
{
  const auto it = g_args.find(key);
  return it == g_args.end() ? otherwise : it->second;
}

const char *name_of(const void *kernel)
{
  Dl_info info{};
  return kernel && dladdr(kernel, &info) && info.dli_sname ? info.dli_sname : "-";
}

umpa_fr_settings settings()
{
  umpa_fr_settings s{};
  s.interpolation = arg("evaluated") || arg("nearest") ? UMPA_FR_DYNAMIC : UMPA_FR_LOOKUP;
  s.type = arg("nearest") ? UMPA_FR_FAST : UMPA_FR_PRECISE;
  s.alpha = 15.f;
  s.blobRadius = (float)arg("radius", 1.9);
  return s;
}

void insert()
{
  const int box = (int)arg("box"), side = box + 1, spaces = (int)arg("spaces", 1);
  const umpa_fr_settings s = settings();
  umpa::FrVariant v{};
  v.mode = arg("nearest") ? umpa::kModeNearest
           : arg("evaluated") ? umpa::kModeFastKaiser : umpa::kModeLookup;
  v.nb = umpa::host::footprint(s);
  v.half = arg("half") != 0;
  v.fastMath = v.half || arg("fast") != 0;
  v.count = arg("count") != 0;
  v.batched = arg("batched") != 0;
  v.kernel = (int)arg("kernel");
  v.tableGlobal = arg("tableGlobal") != 0;
  umpa::FrJob job{};
  job.xSize = box / 2 + 1;
  job.ySize = box;
  job.sliceElems = (int64_t)job.xSize * job.ySize;
  job.nProj = (int)arg("slices", spaces);
  job.vx = job.vy = job.vz = side;
  job.spaceEnd = spaces;
  job.shiftBox = umpa::host::box_can_shift(s, (uint64_t)job.xSize, (uint64_t)job.ySize);
  job.c.cBlobRadius = s.blobRadius;
  v.shift = job.shiftBox != 0;
  umpa::FrLaunch l{};
  l.nTable = (int)arg("table", 10000);
  l.waveItems = (int)arg("waveItems");
  if (!v.batched && umpa::cells_possible(side, side, side)) {
    l.cellsShared = umpa::host::share_cells(side, side, side, (uint64_t)spaces, s);
    l.nCells = (int)umpa::host::make_cell_blocks(side, side, side, l.cellsShared).size() / 2;
  }
  const float core = v.batched || v.fastMath ? 0.f : umpa::host::core_radius(side, side, side);
  l.nItems = (int)umpa::host::make_brick_schedule(side, side, side, v.fastMath, {}, core).size();
  if (core > 0.f) l.nCore = (int)umpa::host::core_cells(side, side, side, core).size() / 2;
  const umpa::FrChoice c = umpa::choose_fr_insert(job, l, v, (int)arg("cus", 256));
  std::printf("%d %d %d %zu %s\n", c.which, c.blocks, c.threads, c.lds, name_of(c.kernel));
}

void batch_tuner()
{
  const bool half = arg("half") != 0, fast = half || arg("fast") != 0;
  const auto schedules = umpa::host::batch_tuning_candidates(
    fast, umpa::host::batch_auto_kernel(fast, half, arg("bounded") != 0));
  std::printf("%d,%d", schedules[0].kernel, schedules[0].boxFixed ? 1 : 0);
  for (const auto &c : umpa::host::batch_kernel_candidates(schedules[0], fast))
    std::printf(" %d,%d", c.kernel, c.boxFixed ? 1 : 0);
  std::printf(" %zu\n", schedules.size());
}

void op_tuner()
{
  const bool half = arg("half") != 0, fast = half || arg("fast") != 0;
  for (const auto &c : umpa::host::op_tuning_candidates(fast, half, arg("cells") != 0))
    std::printf("%d ", c.kernel);
  std::printf("\n");
}

void op_key()
{
  const int side = (int)arg("box") + 1;
  const bool half = arg("half") != 0, fast = half || arg("fast") != 0;
  const umpa_fr_settings s = settings();
  const uint64_t spaces = (uint64_t)arg("spaces"), init = (uint64_t)arg("init", arg("spaces"));
  std::printf("%s\n", umpa::host::op_tuning_key(
                        256, umpa::kModeLookup, fast, half, umpa::host::footprint(s), side, spaces,
                        umpa::host::plain_depth_scale(side, side, side, init, s, fast),
                        umpa::host::share_cells(side, side, side, init, s)).c_str());
}

void batch_key()
{
  const bool half = arg("half") != 0, fast = half || arg("fast") != 0;
  std::printf("%s\n", umpa::host::batch_tuning_key(
                        256, umpa::kModeLookup, fast, half, umpa::host::footprint(settings()),
                        arg("bounded") != 0,
                        { { (int)arg("box") + 1, (int)arg("spaces") } }).c_str());
}

void core()
{
  const int side = (int)arg("box") + 1;
  const float radius = umpa::host::core_radius(side, side, side);
  std::printf("%zu %zu\n", umpa::host::core_cells(side, side, side, radius).size() / 2,
              umpa::host::make_brick_schedule(side, side, side, false, {}, radius).size());
}

void depth()
{
  const int side = (int)arg("box") + 1;
  const bool split = arg("fast") != 0;
  std::printf("%g %g\n",
              umpa::host::batch_depth_scale(side, side, side, arg("bounded") != 0, split),
              umpa::host::plain_depth_scale(side, side, side, 1000, settings(), split));
}

}  // namespace

int main()
{
  std::string line;
  while (std::getline(std::cin, line)) {
    std::istringstream is(line);
    std::string command, word;
    is >> command;
    g_args.clear();
    while (is >> word) {
      const size_t eq = word.find('=');
      g_args[word.substr(0, eq)] = eq == std::string::npos ? 1 : std::stod(word.substr(eq + 1));
    }
    if (command == "insert") insert();
    else if (command == "batch_tuner") batch_tuner();
    else if (command == "op_tuner") op_tuner();
    else if (command == "op_key") op_key();
    else if (command == "batch_key") batch_key();
    else if (command == "core") core();
    else if (command == "depth") depth();
    else return 2;
  }
  return 0;
}
