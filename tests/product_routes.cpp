/*
 * Prints what the dispatch rules of the products decide on a card of 256 compute units, without a device: one line per line of the input,
 *   plain <element size> <matrices> <rows> <columns> <bytes of a K row>      "<tiles 0|1> <by rows 0|1> <direct kernel 0|1> <tile>"
 *   dense ...                                                                "<tiles 0|1> 0 <direct kernel 0|1> <tile>"   (bias, no C)
 *   residual ...                                                             the same with C
 *   experts ...                                                              as dense, with the matrices' rows side by side
 *   through ...                                                              "<write-through 0|1>" of a batch of plain products
 *   straddling <element size> <bytes of a pixel> <pixels> <columns> <bytes of a K row>      "<register-staged 0|1>"
 */
#include "conv_tiles.hpp"
#include "gemm_direct.hpp"

#include <cstdio>
#include <cstring>

namespace mlhip
{
	int device_compute_units()
	{
		return 256;
	}
}

int main()
{
	char kind[16];
	int element_size;
	mlhip::StreamGemmArgs g { };
	while (std::scanf("%15s %d %d %d %d %d", kind, &element_size, &g.batch, &g.M, &g.N, &g.k_bytes) == 6)
	{
		if (std::strcmp(kind, "straddling") == 0)
		{
			mlhip::ConvTileArgs c { };
			c.c_bytes = g.batch;
			c.M = g.M;
			c.N = g.N;
			c.k_bytes = g.k_bytes;
			std::printf("%d\n", mlhip::stays_register_staged(c, element_size));
			continue;
		}
		if (std::strcmp(kind, "through") == 0)
		{
			g.a_row_bytes = 0;
			std::printf("%d\n", mlhip::products_write_through(g, element_size));
			continue;
		}
		const bool plain = std::strcmp(kind, "plain") == 0;
		g.a_row_bytes = (std::strcmp(kind, "experts") == 0) ? static_cast<size_t>(g.batch) * g.k_bytes : 0;
		const mlhip::GemmTile tile = plain ? mlhip::tile_of_plain(g, element_size) : mlhip::tile_with_epilogue(g, element_size);
		const char *names[] = { "64x64", "128x64", "128x128", "128x192" };
		std::printf("%d %d %d %s\n", plain ? mlhip::plain_gemm_tiles_apply(g, element_size) : mlhip::gemm_tiles_apply(g, element_size, std::strcmp(kind, "residual") == 0),
				plain && mlhip::products_go_by_rows(g, element_size), element_size == 2 && mlhip::gemm_direct_applies(g), names[static_cast<int>(tile)]);
	}
	return 0;
}
