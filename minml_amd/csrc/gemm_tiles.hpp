/*
 * gemm_tiles.hpp — batched products C[i] = A[i] * B[i]^T (plain store) whose rows are too many for the direct kernel (gemm_direct.hpp) and too
 * few for the streaming one (gemm_stream.hpp): the 36 Winograd products of about ten to two hundred positions, and every number of rows
 * for the K rows and types that have no kernel of their own (fp32; K rows of any multiple of 64 bytes).
 *
 * A streaming workgroup spends about 10 us on its B operand and its first stages before it multiplies, which a launch of 20 us does not get
 * back, and the tile engine's pipeline is longer than these rows. Here a workgroup owns one tile of 64 to 128 rows and 64 to 192 columns and walks
 * K in pieces of 128 bytes through two LDS slots; two to four workgroups share a compute unit and cover one another's round trips, and
 * the grid hands out tiles as they finish. 32x32 MFMA blocks in the order of K of the other engines: bit-identical to them, so that a
 * position's result does not depend on its batch.
 *
 * What bounds it is where its operands lie. Each XCD has its own L2 (8 x 4 MB), and what a launch has written there the next one finds, if
 * the workgroup that wants it runs on the same XCD: the order of the grid decides. By matrix, an XCD works on a few of the matrices and
 * fetches all their rows. By rows, it works on one eighth of the rows of ALL matrices, the eighth that the transforms before and after
 * it handle on the same XCD (winograd.hip): A comes from this L2 and C stays in it, at the price of every XCD fetching all of B.
 *
 * Measured in networks (40 layers with weights of their own, us per product + fused transform; before: streaming or direct product, in
 * fp32 from 192 channels on the tile engine, and transforms that send the images round the XCDs):
 *   fp16  64 channels (direct kernel by rows) 1024 rows 15.2 -> 12.0; 128 channels 512 rows 15.5 -> 12.1, 1616 24.2 -> 19.9, 4096 35.3 -> 33.7;
 *         192 channels 640 rows 21.9 -> 17.9, 4096 61.3 -> 57.5; 256 channels 256 rows 16.4 -> 15.2, 640 26.1 -> 21.3, 1616 39.1 -> 36.7;
 *         384 channels 256 rows 23.7 -> 20.0, 832 47.2 -> 36.3, 2304 79.6 -> 73.7
 *   fp32  64 channels 16 rows 10.8 -> 7.8, 512 17.1 -> 10.7; 128 channels 64 rows 19.7 -> 10.2, 512 25.7 -> 19.8, 4096 82.4 -> 77.2;
 *         256 channels 64 rows 18.5 -> 14.9, 512 48.5 -> 39.0, 2048 200 -> 113
 * and alone, the stem's products (K = 32, fp16, 256 columns): 64 rows 5.7 -> 3.7, 1616 12.7 -> 10.6, 8192 32.4 -> 30.1.
 */
#ifndef MINML_AMD_GEMM_TILES_HPP_
#define MINML_AMD_GEMM_TILES_HPP_

#include "common.hpp"
#include "epilogues.hpp"
#include "gemm_stream.hpp"

namespace mlhip
{
	/* what the products read once and write: all of A and C. Limits and figures in MB of 10^6 bytes */
	constexpr unsigned long long MB = 1000 * 1000;
	inline unsigned long long exchanged_bytes(const StreamGemmArgs &g, int element_size)
	{
		return static_cast<unsigned long long>(g.batch) * g.M * (static_cast<unsigned long long>(g.k_bytes) + static_cast<unsigned long long>(g.N) * element_size);
	}
	/*
	 * Whether the transforms before and after a batch may divide its rows among the XCDs: the 36 matrices of their 6x6 tiles. Any other batch gains nothing
	 * from the order by rows and pays for it, each XCD fetching all of B; and so do 36 matrices with many more columns than rows. Alone, fp16, us by
	 * matrix / by rows: 16 x 512 x 2048, 128-byte K rows (streaming kernel) 11.5 / 16.6, 64 x 192 x 1024 9.8 / 13.5; 64 x 192 x 1024, 256 bytes 13.4 / 14.6, 512
	 * 16.6 / 20.9; 16 x 1024 x 1024, 512 bytes 17.0 / 20.9; 36 x 192 x 1024, 384 bytes 10.8 / 11.5.
	 */
	constexpr int TRANSFORM_MATRICES = 36;
	inline bool between_transforms(const StreamGemmArgs &g)
	{
		return g.batch == TRANSFORM_MATRICES && g.N <= 2LL * g.M;
	}
	/*
	 * By rows (header) while A and C fit the L2s of the XCDs and there are enough rows to divide among them. us per product + transform, 64x64
	 * tiles by matrix / by rows: fp16 256 channels 128 rows 11.0 / 11.0, 192 12.9 / 12.8, 256 15.5 / 15.2, 384 19.5 / 18.0; 128 channels 256 rows 10.1 / 9.8, 1024
	 * 21.0 / 15.5, 2048 (38 MB) 23.2 / 22.0; tiles of 128x64: 256 channels 960 rows (35 MB) 27.9 / 27.1, 1152 (42 MB) 31.8 / 31.7, 1408 35.5 / 35.0, 2304 52.2 / 51.8;
	 * 384 channels 640 rows (35 MB) 31.0 / 30.1, 768 (42 MB) 36.1 / 35.8, 1024 41.2 / 42.3; fp32 128 channels 160 rows 12.3 / 12.2, 192 13.0 / 12.5, 1024 (38 MB)
	 * 29.7 / 27.2, 1616 (60 MB) 39.7 / 39.7.
	 */
	inline bool products_meet_in_l2(const StreamGemmArgs &g, int element_size)
	{
		return between_transforms(g) && g.M >= 192 && exchanged_bytes(g, element_size) <= 42 * MB;
	}
	/*
	 * And beyond where all of B takes a small part of each L2, while the transforms divide the images like that (matrices_stay_cached in
	 * winograd.hip). With weights that come from memory (200 layers): fp16 128 channels (1.2 MB), 4096 rows 38.6 / 34.7; fp32 128 channels (2.4 MB), 1616 rows
	 * 41.2 / 39.9; level with 40 layers, and behind with 2.7 MB (fp16, 192 channels, 2560 rows 36.3 / 37.9).
	 */
	inline bool products_go_by_rows(const StreamGemmArgs &g, int element_size)
	{
		const unsigned long long b_bytes = static_cast<unsigned long long>(g.batch) * g.N * g.k_bytes;
		return products_meet_in_l2(g, element_size)
				|| (between_transforms(g) && g.M >= 8 * static_cast<long long>(g.N) && 5 * b_bytes <= 13 * MB && exchanged_bytes(g, element_size) <= 117 * MB);
	}
	/*
	 * Whether these tiles take a batch of plain products, by the number of 32x32 tiles and the bytes of A and C (figures as above, other
	 * kernel / this one).
	 * Not where the direct kernel's 32x32 tiles are few enough to be ahead: 256-byte rows, 128 channels, 448 rows (2016 tiles) 13.0 / 14.1 us, 512 (2304) 12.9 /
	 * 12.1; 512: 256 channels, 96 rows (864) 10.4 / 10.7, 128 (1152) 11.3 / 11.0; 384: 192 channels, 96 rows (648) 9.0 / 9.4, 160 (1080) 10.6 / 10.5; 768: 384
	 * channels, 32 rows (432) 10.5 / 11.2, 64 (864) 13.0 / 12.2. Other batches than the 36 of a network gain nothing around the product (alone): 512 bytes,
	 * 8 x 400 x 400 (1352) 4.5 / 5.0, 100 x 128 x 128 (1600) 4.8 / 5.1, 16 x 400 x 400 (2704) 6.6 / 6.6, 24 x 512 x 256 (3072) 6.8 / 6.2; 768, 16 x 192 x 256 (768) 4.7 / 5.2,
	 * 64 x 128 x 128 (1024) 5.5 / 5.0. And fp32 rows of 384 bytes and more but 512, for which the small tiles of conv_tiles.hpp stand,
	 * resident at once to one per unit: 192 channels, 32 rows (216) 10.7 / 11.6, 64 (432) 13.8 / 12.2; alone, 8 x 512 x 64 (256) 640 bytes 5.5 / 6.2, 768 5.5 / 6.9, 896 6.3 / 7.5, 8 x 600 x 64 (304)
	 * 6.5 / 6.2, 6.5 / 6.9, 7.6 / 7.6, to 512 the same, then 8.3 / 6.4, 9.1 / 7.0, 10.0 / 7.7. From 1024 bytes on they stand to two per unit, the most that conv_tiles.hpp gives them, and
	 * the more K the further they are ahead (alone): 36 x 16 x 256 (288) 8.0 / 8.6, 36 x 16 x 384, 1536 bytes (432) 10.9 / 12.0, 9 x 776 x 56, 2048 bytes
	 * (450) 13.5 / 14.8, 8 x 64 x 512, 4096 bytes (256) 17.0 / 25.2, 8192 (256) 30.1 / 46.4, 8 x 128 x 512 (512) 41.9 / 46.8, 16384 78.3 / 89.6; above, 36 x 64 x 256 (576, in a
	 * network) 18.5 / 14.9.
	 * fp16 rows of one, two or three pieces and a half beyond 252 MB only with one or three column tiles (this one's time over the other's, 36 matrices): 192 bytes 256 columns 200 MB 0.88, 300 1.06, 700 1.06,
	 * 128 columns 0.76, 1.08, 1.06, 384 columns 0.79, 0.97, 0.99, 64 0.73, 0.79, 0.81; 320 bytes 256 columns 0.86, 1.06, 1.07, 512 0.90, 1.02, 1.04, 384 0.79, 0.94, 0.88; 448 bytes 256 columns 0.87,
	 * 1.02, 1.03, 512 0.91, 1.04, 1.02, 128 0.84, 0.96, 0.98.
	 * Other K rows have no limit in bytes: what else would take them is behind throughout (other kernel / this one): fp16 36 x 11815 x 64, 576 bytes (299 MB) 72.1 / 60.4, 36 x 17871 x 256 (700)
	 * 236 / 209, 36 x 16113 x 512, 640 (965) 564 / 355, 36 x 15990 x 256, 704 (700) 242 / 212, 36 x 21701 x 256, 384 (700) 260 / 210; fp32 64 x 3512 x 256, 768 (403) 284 /
	 * 202, 8 x 4741 x 512, 1024 (117) 169 / 92, 36 x 3425 x 384, 1536 (379) 334 / 316, 36 x 7479 x 128 (551) 288 / 235, 4 x 15450 x 1024 (348) 485 / 417, 64 x 4248 x 192, 2048 (766) 529 / 458.
	 * Not beyond a number of bytes where the streaming kernel, which fetches A once, or for 64 and 128 bytes the kernels that store more at
	 * a time are level or ahead: fp16 256-byte rows 57 MB 32.2 / 28.8, 75 35.3 / 33.7, but with three calls per layer 23.6 / 24.0 and 94 MB 28.3 / 29.5; 512: 94 MB 53.3 / 53.3, 113 59.1 / 61.4, 302 127 / 143; 768, of
	 * which the streaming kernel holds only 128 columns (whole networks of 8 blocks, 384 channels): 239 MB 2352 / 2083, 292 2706 / 2499, but with three
	 * calls per layer 265 MB 2435 / 2472, where three or five column tiles leave its slices of 128 columns padded or some compute units idle; other widths, alone
	 * (12 and 36 matrices, this one's time over the other's): 256 columns 150 MB 0.96, 200 1.05, 245 1.16, 512 150 0.96, 200 0.99, 245 1.13, 1024 90 0.85, 120 0.95, 200 1.04, 245 1.20 (64 matrices 108 1.06),
	 * 2048 150 1.03, 245 1.18; 320 245 0.88, 640 0.90). Other batches than the 36 of a network have their operands as often from memory (cached / from memory, 16 matrices):
	 * 256 bytes to 34 MB, 24 MB 128 columns 0.70 / 0.92, 256 0.83 / 1.05, 512 0.78 / 0.93, 32 0.82 / 1.06, 0.82 / 1.08, 0.74 / 1.01, 54 0.83 / 1.11, 0.83 / 1.20, 0.94 / 1.36;
	 * 512 to 67, 256 columns 66 MB 0.76 / 0.95, 80 0.82 / 1.05, 92 0.86 / 1.12, 1024 columns 66 0.74 / 0.96, 80 0.97 / 1.30; 768 to 105, 256 columns 92 0.82 / 1.05, 130 0.87 / 1.10, 512 92 0.74 / 0.96,
	 * 130 0.83 / 1.07, beyond 512 columns to 84, 1024 80 0.76 / 0.96, 92 0.96 / 1.22, in three or five column tiles to 210, 384 200 0.76 / 0.97, 250 0.85 / 1.07, 640 200 0.92 / 1.10, 250 1.02 / 1.14. fp32 256-byte rows, where those slices are not padded by more than an eighth: 128 columns 250 MB 0.94, 300 1.00,
	 * 450 1.06, 256 columns 250 0.98, 300 1.08, 450 1.13, 512 250 1.03, 300 1.09, 600 1.18 (64 columns 600 MB 0.92, 192 0.88); fp32 512-byte rows 151 MB 82.4 / 79.9, 227
	 * 117 / 123; 64-byte rows (the stem, alone) 170 MB 32.4 / 29.3, 340 89.8 / 101; fp32 128-byte rows, the stem, with the
	 * input from memory 24 MB 11.9 / 10.1, 47 16.6 / 16.4, 57 16.6 / 17.7, 85 23.3 / 27.6, 94 23.3 / 27.6; whole networks of one block 128 channels 9 MB 67.2 / 63.9, 38
	 * 125.3 / 125.3, 47 144.9 / 144.5, 66 184.3 / 185.4, 94 241.3 / 245.6, 256 channels 42 MB 195.3 / 194.6, 67 276.8 / 280.6, 64 channels, for
	 * which A is fetched once, 57 MB 124.8 / 123.6, 111 200.3 / 204.6.
	 */
	inline bool plain_gemm_tiles_apply(const StreamGemmArgs &g, int element_size)
	{
		const bool fp16 = element_size == 2, between = g.batch == TRANSFORM_MATRICES;
		if (g.k_bytes % 64 != 0 || (fp16 && (g.k_bytes == 128 || g.k_bytes > 768)))
			return false;
		const long long tiles = static_cast<long long>(ceil_div(g.M, 32)) * ceil_div(g.N, 32) * g.batch;
		long long fewest = 0; /* 32x32 tiles per compute unit */
		unsigned long long megabytes = ~0ULL / MB; /* most of A and C together */
		switch (g.k_bytes)
		{
			case 64:
				megabytes = 283;
				break;
			case 128:
				megabytes = (g.N <= 64) ? 63 : 50;
				break;
			case 256:
				fewest = fp16 ? 8 : 0;
				if (fp16)
					megabytes = between ? 67 : 34;
				else if (g.N > 64 && 8 * (ceil_div(g.N, 128) * 128LL - g.N) <= g.N)
					megabytes = 268;
				break;
			case 384:
				fewest = fp16 ? 4 : 1;
				break;
			case 512:
				fewest = fp16 ? (between ? 4 : 8) : 0;
				megabytes = fp16 ? (between ? 94 : 67) : 210;
				break;
			case 768:
				fewest = fp16 ? (between ? 3 : 4) : 1;
				if (fp16 && (ceil_div(g.N, 64) % 3 == 0 || ceil_div(g.N, 64) % 5 == 0) && g.N <= 1024)
					megabytes = between ? 252 : 210;
				else if (fp16)
					megabytes = (g.N <= 512) ? (between ? 168 : 105) : (between ? 105 : 84);
				break;
			case 192:
			case 320:
			case 448:
				fewest = (fp16 || g.k_bytes < 384) ? 0 : 1;
				if (fp16 && g.N > 64 && ceil_div(g.N, 64) % 3 != 0)
					megabytes = 252;
				break;
			default:
				fewest = (fp16 || g.k_bytes < 384) ? 0 : 1;
				break;
		}
		if (!fp16 && g.k_bytes >= 384 && g.k_bytes % 128 == 0 && g.k_bytes != 512 && tiles <= (g.k_bytes >= 1024 ? 2LL : 1LL) * device_compute_units())
			return false;
		return tiles >= fewest * device_compute_units() && exchanged_bytes(g, element_size) <= megabytes * MB;
	}
	/*
	 * The same for products with bias (+ beta * C), linear or ReLU: dense layers, 1x1 convolutions, the experts' layers. Alone, other kernel / this one, us, and
	 * the number of 64x64 tiles:
	 *   fp16, from 1.75 tiles per unit with rows up to 512 bytes (256 x 256: 2700 rows (172) 4.3 / 4.8, 7200 (452) 5.7 / 5.6; 128 to 768: 2700
	 *   (516) 5.9 / 5.2), 1 up to 768 bytes (384 x 256: 7200 (452) 11.0 / 6.5; x 384: 2700 (258) 6.2 / 6.0), 0.5 up to 1024, where the 32x32 tiles of
	 *   conv_tiles.hpp end (512 x 256: 2048 (128) 5.5 / 5.7, from memory 5.2 / 5.9, 2300 (144) 6.9 / 5.8, 2700 (172) 7.0 / 6.0; eight experts 228 rows (128) 5.3 / 5.7, 300
	 *   (160) 6.5 / 5.8). Longer
	 *   rows, for which a tile of 256 rows is the better one where there are enough, to 4 per unit (3 for experts of 2048 bytes and at most 128 columns: eight of 1024 x 128, 3072 rows 15.7 / 13.8, from
	 *   memory 20.8 / 20.2, 3584 17.3 / 17.3 and 23.1 / 24.6; of 768 x 128 16.1 / 14.0 and 19.9 / 20.9; one of 1024 x 128, 28672 rows 20.9 / 17.0 and 25.6 / 24.6) and 8192 bytes of K rows per unit (eight experts of 576 to 2048 x 256,
	 *   from L2: 300 rows (160) 1152 bytes 6.9 / 6.2, 2048 9.7 / 8.9, 4096 15.6 / 13.9; 912 (480) 9.4 / 8.0, 13.2 / 10.7, 21.1 / 17.6; 1824 (928) 13.3 / 12.1, 18.5 /
	 *   17.6, 30.4 / 32.1, from memory 14.3 / 14.5, 21.8 / 22.1, 37.4 / 39.3; 2100 (1056) 14.0 / 14.7, 20.2 / 22.2, 33.6 / 37.1; 3072 bytes 1200 (608) 22.1 / 18.1, 1824 from
	 *   memory 30.2 / 31.7; single layers of 256 columns, whose other kernel has its epilogue at run time, 1536 bytes 10800 rows (676) 13.6 / 10.6, 14400 (900) 15.7 / 14.1). 1024 with a batch to 8 (512 x 1024: 912 rows (1920) 18.5 / 15.9, 3648 (7296) 43.5 / 46.4).
	 *   Half a tile of padding is not for them: at most 32 columns where the streaming or direct kernel take the rows, from 3.5 tiles per unit (28800 x 32: 256-byte
	 *   rows (450) 3.9 / 4.4, 512 4.7 / 5.1, 768 5.5 / 5.9; 57600 (900) 5.2 / 5.3, 7.4 / 7.3, 14.1 / 11.0); 384 bytes, whose direct kernel has no upper limit,
	 *   from 64 columns (114119 x 32 10.8 / 11.9, 230400 x 24 17.3 / 18.9, 57600 x 40 from memory 8.6 / 9.2).
	 *   Not beyond a number of bytes of A, C and what is read of it where the streaming kernel takes the rows: ahead further with the operands in the last-level
	 *   cache than from memory (this one's time over the other's, cached / from memory), and with a residual, whose fetch the other does not hide, further than without.
	 *   256-byte rows to 34 MB: 128 columns 32 MB 0.77 / 0.94, 40 0.87 / 1.05, 66 0.92 / 1.12; 256 columns 24 0.87 / 1.05, 32 0.85 / 1.06, 40 0.97 / 1.22, 95 1.00 / 1.38; 1024
	 *   columns 24 0.82 / 0.99, 40 0.89 / 1.15, 80 1.04 / 1.47. 512 to 46 MB: 256 columns 40 MB 0.77 / 0.97, 52 0.91 / 1.09, 95 0.94 / 1.19; 1024 columns 40 0.85 / 1.05, 52 0.90 /
	 *   1.18, 80 1.04 / 1.36. 768 to 67 MB: 256 columns 66 MB 0.79 / 1.02, 95 0.84 / 1.09; 1024 columns 66 0.85 / 1.04, 80 0.86 / 1.10. With a residual to 101 MB: 256-byte rows 40
	 *   to 95 MB 0.87 to 1.04 / 0.86 to 1.11, 512 0.80 to 0.93 / 0.80 to 1.06, 768 0.80 to 0.95 / 0.87 to 1.07 (256 x 256: 57600 rows, 88 MB with residual, 26.4 / 23.8,
	 *   115200 (177) 41.7 / 41.7, 230400 81.5 / 105; 256 x 1024: 27797 (71) 28.7 / 28.1, 57600 (147) 48.8 / 55.1; 384 x 384 with residual: 27797 (64) 25.2 / 22.2, 57600
	 *   (133) 39.7 / 40.1; eight experts of 256 x 1024: 7296 rows (149) 57.1 / 55.4, 14592 89 / 127), to 189 with at most 128 columns
	 *   from 512 bytes on (512: 66 to 130 MB 0.81 / 1.06 to 0.80 / 1.04, 768 130 MB 0.75 / 1.00; with residual 256 bytes 230400 rows (177) 36.4 / 34.2, 369664 (284) 50.2 / 68.8, but
	 *   from memory 130 MB 0.95 / 1.08).
	 *   fp32, rows of 256 and 512 bytes, which only the streaming kernel took: always (128 x 128: 225 rows 17.2 / 6.2, 27797 20.2 / 16.4, 230400 105 / 87); those of
	 *   experts (a_row_bytes), for which the 32x32 tiles of conv_tiles.hpp stand, from where these end (eight of 128 x 64: 64 rows 4.5 / 5.6, 512 4.7 / 5.7, 800 5.4 / 5.8; 36 of 64 x 64: 85 rows
	 *   3.8 / 4.3, 177 4.3 / 4.4; sixteen of 128 x 256, 809 rows 16.2 / 14.2).
	 *   Others up to 4096 bytes from 0.6 (256 x 256: 900 rows (60) 6.8 / 8.8, 2700 (172) 11.8 / 9.2, 57600 87.6 / 74.5).
	 */
	inline bool gemm_tiles_apply(const StreamGemmArgs &g, int element_size, bool reads_c)
	{
		const long long tiles = static_cast<long long>(ceil_div(g.M, 64)) * ceil_div(g.N, 64) * g.batch, units = device_compute_units();
		const long long small_tiles = static_cast<long long>(ceil_div(g.M, 32)) * ceil_div(g.N, 32) * g.batch;
		if (g.k_bytes % 64 != 0)
			return false;
		if (element_size == 4 && (g.k_bytes == 256 || g.k_bytes == 512))
			return g.a_row_bytes == 0 || small_tiles > 2 * units;
		if (element_size == 4)
			return g.k_bytes <= 4096 && 8 * tiles >= 5 * units;
		if (g.k_bytes < 192 || (g.k_bytes > 768 && g.k_bytes % 128 == 0 && small_tiles <= 2 * units))
			return false;
		if (g.k_bytes > 1024)
			return g.k_bytes <= 4096 && small_tiles > 2 * units && tiles <= ((g.batch > 1 && g.N <= 128 && g.k_bytes >= 2048) ? 3 : 4) * units && tiles * g.k_bytes <= 8192 * units;
		if (g.k_bytes > 768 && g.batch > 1 && tiles > 8 * units)
			return false;
		const bool streams = g.k_bytes == 256 || g.k_bytes == 512 || g.k_bytes == 768;
		const unsigned long long bytes = exchanged_bytes(g, element_size) + (reads_c ? static_cast<unsigned long long>(g.batch) * g.M * g.N * element_size : 0);
		if ((g.k_bytes == 384 && g.N < 64) || (streams && g.N <= 32 && 2 * tiles < 7 * units))
			return false;
		const unsigned long long megabytes = (g.N <= 128 && g.k_bytes > 256) ? 189 : reads_c ? 101 : g.k_bytes == 256 ? 34 : g.k_bytes == 512 ? 46 : 67;
		return 4 * tiles >= (g.k_bytes <= 512 ? 7 : g.k_bytes <= 768 ? 4 : 2) * units && !(streams && bytes > megabytes * MB);
	}
	/* rows x columns of the tile that a workgroup owns */
	enum class GemmTile
	{
		T64x64, T128x64, T128x128, T128x192
	};
	/*
	 * Whether 128 rows to a tile pad at most a quarter more than 64 do. Short matrices of a batch, or a few rows and many columns, would be multiplied twice:
	 * fp16, us, 64x64 / 128x64 / 128x128: 64 x 16 x 1024, 256-byte K rows 5.1 / 6.6 / 5.8; 48 x 22 x 2000, 384 bytes 9.5 / 10.7 / 10.6 (direct kernel
	 * 8.9); 64 x 64 x 1024 7.1 / 9.2 / 8.1 (7.7); 32 x 190 x 2048, 256 bytes 11.9 / 13.3 / 11.8 (12.8); 64 x 70 x 1024, 512 bytes, which both pad to
	 * 128, 11.5 / 10.9 / 9.9; one of 40 x 60000 with ReLU, 384 bytes 6.7 / 9.4 / 7.9 (6.6).
	 */
	inline bool fills_128_rows(const StreamGemmArgs &g)
	{
		return 8LL * ceil_div(g.M, 128) <= 5LL * ceil_div(g.M, 64);
	}
	/*
	 * Plain products: larger tiles, which fetch less, once there are enough of them and M fills them. fp16 by rows, 64x64 / 128x64: 256 channels 448 rows (1008 tiles of 64x64) 18.6 / 19.2, 512
	 * (1152) 19.8 / 19.1; 128 channels 896... 960 rows (1080) 16.1 / 16.0; 384 channels 192 rows (648) 18.9 / 19.4, 256 (864) 21.6 / 20.6. By matrix, 128x64 / 128x128:
	 * 192 channels 2304 rows 32.8 / 35.5; 256 channels 1616 rows 37.8 / 36.7, 2304 52.2 / 51.2; 384 channels 1408 rows 58.4 / 55.1, 3072 97.5 / 95.6. fp32 stays at
	 * 64x64: 128 channels 2048 rows 45.6 / 46.0, 256 channels 960 63.0 / 65.5, 640 46.7 / 45.8 (128x64).
	 * By matrix tiles of 128x192 wherever they pad the columns no more than 64 would: A is fetched once for 192 columns and twice for 384, in place of
	 * three times by either of the others, and nothing is multiplied for padding as by 128x128 at 192. Whole networks, the tile before / this one, us: 192
	 * channels, 10 blocks, 1616 rows 640 / 599, 4800 1401 / 1383, with three calls per layer (8 blocks) 1616 564 / 538, 6400 1540 / 1435; 384 channels, 1024 rows
	 * 856 / 827, 1616 1225 / 1200, 2880 1957 / 1898, with three calls per layer 3248 1734 / 1679. By rows they are level or behind, with too few of
	 * them for two rounds (8 blocks: 192 channels 768 rows 333.5 / 337.2, 384 channels 256 rows 352.2 / 356.5), and as a dense layer with its epilogue, whose
	 * side inputs do not fit the registers beside three blocks (192 channels with residual, 184832 rows 57.7 / 67.0, 384 channels 27797 21.1 / 21.9).
	 */
	inline GemmTile tile_of_plain(const StreamGemmArgs &g, int element_size)
	{
		const long long tiles = static_cast<long long>(ceil_div(g.M, 64)) * ceil_div(g.N, 64) * g.batch;
		if (element_size != 2 || tiles < (g.k_bytes >= 768 ? 3 : 4) * device_compute_units() || !fills_128_rows(g))
			return GemmTile::T64x64;
		const bool by_rows = products_go_by_rows(g, element_size);
		if (!by_rows && ceil_div(g.N, 64) % 3 == 0)
			return GemmTile::T128x192;
		return (!by_rows && g.k_bytes >= 512) ? GemmTile::T128x128 : GemmTile::T128x64;
	}
	/*
	 * Whether the 36 products between transforms write through the L2 (store_through_l2 in device_utils.hpp), so that the transform after them does not wait until they are
	 * written back. Networks of 20 blocks, us, written back / through: fp16 256 channels 15x15 12 positions 492 / 469, 16 535 / 520 (with weights that come from memory 560 / 564), 32 755 / 735, 19x19 8 609 / 590, 32 993 / 974; 128
	 * channels 32 424 / 413, 64 600 / 576, 101 827 / 832, 19x19 100 1186 / 1142; 192 channels 16 448 / 433, 64 884 / 874; 64 channels 64 405 / 405; 384 channels 8 583 / 574, 64 1623 / 1608; fp32 64 channels
	 * 32 444 / 441, 128 channels 32 751 / 713, 64 1124 / 1080, 256 3325 / 3318, 256 channels 16 1060 / 1019. Not where the launch itself is short of bandwidth to memory: tiles of
	 * 128x128 (256 channels 64 1116 / 1134, 101 1526 / 1574), and orders by rows, in which every XCD fetches all of B, with a large B (384 channels, 10.6 MB, 16 802 / 816, 32 1161 / 1200; the line lies
	 * between 256 and 320 channels, 4.7 and 7.4 MB: two layers of 320, 15x15 12 30.0 / 29.6, 32 50.2 / 50.5, 48 62.6 / 63.6, 19x19 24 55.5 / 56.3).
	 * Rows of C that are not whole lines of 128 bytes leave the L2 in parts: no matter while there are few of them (18 blocks of 96 channels, C of 1.8 MB 430 / 415, 3.5 446 / 440,
	 * 7.1 586 / 583), more traffic than the wait costs after that (19x19, 11 MB 758 / 815; 14 MB 813 / 880, 24 MB 1179 / 1229).
	 */
	inline bool products_write_through(const StreamGemmArgs &g, int element_size)
	{
		if (g.batch != TRANSFORM_MATRICES)
			return false;
		const unsigned long long c_row = static_cast<unsigned long long>(g.N) * element_size;
		if (c_row >= (1ULL << 24) || (c_row % 128 != 0 && c_row * g.batch * g.M > 8 * MB)) /* 128 rows lie within a buffer's 2^31 bytes */
			return false;
		if (element_size == 4)
			return true;
		const unsigned long long b_bytes = static_cast<unsigned long long>(g.batch) * g.N * g.k_bytes;
		return tile_of_plain(g, element_size) != GemmTile::T128x128 && !(products_go_by_rows(g, element_size) && b_bytes > 6 * MB);
	}
	/*
	 * With the epilogue, fp16: 128x128 tiles from 3.5 of 64x64 per unit on (256 x 256, 14400 rows (900): 8.0 / 7.3 us; 384 x 256, 7200 rows (452) 6.5 / 7.7, 14400 9.7 / 8.7), 128x64
	 * where 128 pads the columns more (192 x 192, 57600 rows 15.3 / 14.1).
	 */
	inline GemmTile tile_with_epilogue(const StreamGemmArgs &g, int element_size)
	{
		const long long tiles = static_cast<long long>(ceil_div(g.M, 64)) * ceil_div(g.N, 64) * g.batch;
		if (element_size != 2 || g.k_bytes > 1024 || 2 * tiles < 7 * device_compute_units() || !fills_128_rows(g))
			return GemmTile::T64x64;
		return (ceil_div(g.N, 64) % 2 != 0) ? GemmTile::T128x64 : GemmTile::T128x128;
	}
	/* false: nothing was launched. Plain batched products of fp16 or fp32; and products with bias (+ beta * C), linear or ReLU */
	bool try_launch_gemm_tiles(hipStream_t stream, mlDataType_t dtype, const StreamGemmArgs &g);
	bool try_launch_gemm_tiles(hipStream_t stream, const StreamGemmArgs &g, const FloatEpilogue<half_t> &epilogue);
	bool try_launch_gemm_tiles(hipStream_t stream, const StreamGemmArgs &g, const FloatEpilogue<float> &epilogue);
} /* namespace mlhip */

#endif /* MINML_AMD_GEMM_TILES_HPP_ */
