// The kernels' size rules, evaluated on the host: one form per line of stdin.
//   stage f64 bf16x3 nm nw m0 my nG0 nQuads adaptive mode fuseY learned -> LastStage
//   tiling f64 nm nw nb2max points panels -> mt nt wc rows modes stage lds
//   chunk bytesPerPanel room -> panels
#include <iostream>
#include <string>

#include "../../phoebe_amd/csrc/coupling_tiling.hpp"
#include "../../phoebe_amd/csrc/last_stage.hpp"

int main() {
  std::string kind;
  while (std::cin >> kind) {
    if (kind == "stage") {
      phx::LastStageSizes z{};
      int mode, fuseY, learned;
      std::cin >> z.f64 >> z.bf16x3 >> z.nm >> z.nw >> z.m0 >> z.my >> z.nG0 >> z.nQuads >> z.adaptive >> mode >>
          fuseY >> learned;
      std::cout << int(phx::last_stage(z, mode, fuseY != 0, learned != 0)) << "\n";
    } else if (kind == "tiling") {
      int f64, nm, nw, nb2max, points, panels;
      std::cin >> f64 >> nm >> nw >> nb2max >> points >> panels;
      const phx::CoupTiling c = phx::coupling_tiling(f64 != 0, nm, nw, nb2max, points, panels);
      std::cout << c.mt << " " << c.nt << " " << c.wc << " " << c.rows << " " << c.modes << " " << c.stage << " "
                << c.lds << "\n";
    } else if (kind == "chunk") {
      double per, room;
      std::cin >> per >> room;
      std::cout << phx::panel_chunk(per, std::min(room, phx::kG3RoomMax)) << "\n";
    } else {
      return 1;
    }
    if (!std::cin) return 1;
  }
}
