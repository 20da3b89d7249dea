// Prints host evaluations of functions that the kernels and their launches share.
#include "vector_kernels.hpp"

#include <iostream>
#include <string>

namespace
{
  ppf::GridDesc
  lattice(int n0, int n1, int n2)
  {
    ppf::GridDesc g {};
    g.nodes[0] = n0;
    g.nodes[1] = n1;
    g.nodes[2] = n2;
    return g;
  }

  /// Whether a transfer launch between the lattices is refused, restriction then prolongation.
  std::string
  refused(const ppf::GridDesc &gc, const ppf::GridDesc &gf)
  {
    std::string r;
    for (const ppf::GridDesc *out : {&gc, &gf})
      try
        {
          (void) ppf::transfer_grid(*out, gc, gf, 1);
          r += "0";
        }
      catch (const ppf::Error &)
        {
          r += "1";
        }
    return r;
  }
} // namespace

int
main()
{
  // CG's end flag as the launches with scalars 5, 6 and 7 find it when 6 ends the iteration
  std::cout << "turn_open: " << ppf::cg_ended_before(0, 5) << ppf::cg_ended_before(0, 6) << "\n"
            << "turn_racing: " << ppf::cg_ended_before(6, 6) << "\n"
            << "turn_after: " << ppf::cg_ended_before(6, 7) << "\n"
            << "turn_last_tag: " << ppf::cg_ended_before(0x7fffffff, 1)
            << ppf::cg_ended_before(0x7fffffff, 0x7fffffffu) << "\n";

  // fine planes of just under 2^31 nodes, of 2^31 (the coarse one a quarter), and of
  // 2^33 whose number no 32-bit product holds; more planes than a grid's second extent
  std::cout << "transfer_fits: " << refused(lattice(23170, 23170, 1), lattice(46339, 46339, 1))
            << "\n"
            << "transfer_fine_plane: "
            << refused(lattice(32768, 16385, 1), lattice(65536, 32769, 1))
            << refused(lattice(46341, 46340, 1), lattice(92681, 92679, 1)) << "\n"
            << "transfer_planes: " << refused(lattice(2, 2, 40000), lattice(3, 3, 79999)) << "\n";
}
