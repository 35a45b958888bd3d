// Prints the launch rules of csrc/kernels.h for jobs read from standard input,
// one per line: tw th nr nmu nmus nnu ew iterations iteration half acc64.
// Per job: the SsTiling (block staged nit fixed), its dynamic LDS, fixed_sums,
// sd_split, ms_pairs and ms_spread with the default tile,
// arc_sums.
#include <cstdio>

#include "../../precomputed_atmospheric_scattering_amd/csrc/atmo_device.h"
#include "../../precomputed_atmospheric_scattering_amd/csrc/kernels.h"

int main() {
  atmo::Job j{};
  while (std::scanf("%d %d %d %d %d %d %d %d %d %d %d", &j.tw, &j.th, &j.nr, &j.nmu, &j.nmus,
                    &j.nnu, &j.ew, &j.niter, &j.it, &j.half_luts, &j.acc64) == 11) {
    const atmo::SsTiling t(j);
    j.ms_tile = atmo::ms_default_tile(j.nnu * j.nmus);
    std::printf("%d %d %d %d %zu %d %d %d %d %d\n", t.block, int(t.staged), t.nit, int(t.fixed),
                atmo::ss_lds(j), int(atmo::fixed_sums(j)), atmo::sd_split(j),
                int(atmo::ms_pairs(j)), int(atmo::ms_spread(j)),
                int(atmo::arc_sums(j)));
  }
}
