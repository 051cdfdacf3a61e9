/*
 * gemm_tiles.hpp — batched products C[i] = A[i] * B[i]^T (plain store) whose rows are too many for the direct kernel (gemm_direct.hpp) and too
 * few for the streaming one (gemm_stream.hpp): the 36 Winograd products of about ten to two hundred positions, and every number of rows
 * for the K rows and types that have no kernel of their own (fp32; K rows of any multiple of 64 bytes).
 *
 * A streaming workgroup spends about 10 us on its B operand and its first stages before it multiplies, which a launch of 20 us does not get
 * back, and the tile engine's pipeline is longer than these rows. Here a workgroup owns one tile of 64 or 128 rows and columns and walks
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
#include "gemm_stream.hpp"

namespace mlhip
{
	template<typename T, int BLOCKS_M_, int BLOCKS_N_, int WAVES_M_, int WAVES_N_>
	struct GemmTileShape
	{
			static constexpr int BLOCKS_M = BLOCKS_M_, BLOCKS_N = BLOCKS_N_; /* 32x32 blocks of one wavefront */
			static constexpr int WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, WAVES = WAVES_M * WAVES_N, THREADS = 64 * WAVES;
			static constexpr int BM = 32 * BLOCKS_M * WAVES_M, BN = 32 * BLOCKS_N * WAVES_N;
			static constexpr int SLOTS = 2, SLOT_BYTES = (BM + BN) * 128; /* 128 bytes of K of every row of A and B */
			static constexpr int LOADS = (BM + BN) / 8 / WAVES; /* direct-to-LDS loads (8 rows x 128 bytes) per wavefront and piece */
			static constexpr int SLAB_STRIDE = 32 * BLOCKS_N * static_cast<int>(sizeof(T)) + 16;
			static constexpr int LDS_BYTES = SLOTS * SLOT_BYTES;
			/* workgroups that share a compute unit: as many as the 160 KB of LDS hold, four at most */
			static constexpr int RESIDENT = (160 * 1024 / LDS_BYTES < 4) ? 160 * 1024 / LDS_BYTES : 4;
			static_assert((BM + BN) % (8 * WAVES) == 0, "the same number of loads for every wavefront");
			static_assert(WAVES * 32 * SLAB_STRIDE <= LDS_BYTES, "the slots become the slabs of the store");
	};

	template<typename T, typename Shape>
	__global__ __launch_bounds__(Shape::THREADS, Shape::RESIDENT * Shape::WAVES / 4) void kernel_gemm_tiles_nt(const T *A, const T *B, T *C, int M, int N, int k_bytes,
			size_t stride_a, size_t stride_b, size_t stride_c, unsigned int tiles_m, unsigned int tiles_n, unsigned int matrices, int by_rows)
	{
		typedef MfmaTraits<T> Traits;
		typedef typename Traits::acc_vec acc_vec;
		constexpr int BLOCKS_M = Shape::BLOCKS_M, BLOCKS_N = Shape::BLOCKS_N, WAVES = Shape::WAVES, LOADS = Shape::LOADS;
		const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
		const int wave_m = wave / Shape::WAVES_N, wave_n = wave % Shape::WAVES_N;
		const int frag_row = lane & 31, half_sel = lane >> 5;
		const int pieces = (k_bytes + 127) / 128;

		/* the column tiles of one row tile are neighbours on one XCD; the row tile's matrix changes slowest or its rows do */
		const unsigned int id = xcd_contiguous_block_id(blockIdx.x, gridDim.x);
		const unsigned int row_tile = id / tiles_n;
		const unsigned int slow = row_tile / (by_rows ? matrices : tiles_m);
		const unsigned int fast = row_tile - slow * (by_rows ? matrices : tiles_m);
		const unsigned int matrix = by_rows ? fast : slow;
		const int m_tile = (by_rows ? slow : fast) * Shape::BM, n_tile = (id - row_tile * tiles_n) * Shape::BN;
		const int m0 = m_tile + wave_m * 32 * BLOCKS_M, n0 = n_tile + wave_n * 32 * BLOCKS_N;

		/*
		 * Operands -> LDS slot: [row of A, then of B][128 bytes], the 16-byte chunks of a row swizzled. Rows beyond the matrix repeat its last
		 * row. Row 8 q + 4 h + e of a block of 32 rows of B holds column 16 h + 4 q + e: a lane then ends with 16 consecutive columns.
		 */
		extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
		const uint8_t *a_base = reinterpret_cast<const uint8_t*>(A + matrix * stride_a);
		const uint8_t *b_base = reinterpret_cast<const uint8_t*>(B + matrix * stride_b);
		const uint8_t *src[LOADS];
		static_assert(WAVES % 2 == 0, "the swizzle of a lane is then the same in all its loads");
		const int chunk = ((lane & 7) ^ ((4 * wave + (lane >> 4)) & 7)) * 16;
#pragma unroll
		for (int u = 0; u < LOADS; u++)
		{
			const int row = (wave + WAVES * u) * 8 + (lane >> 3);
			const int place = row - Shape::BM;
			const int column = (place & ~31) + 16 * ((place >> 2) & 1) + 4 * ((place >> 3) & 3) + (place & 3);
			src[u] = ((row < Shape::BM) ? a_base + static_cast<size_t>(min(m_tile + row, M - 1)) * k_bytes
					: b_base + static_cast<size_t>(min(n_tile + column, N - 1)) * k_bytes) + chunk;
		}
		/* the last piece may have 64 bytes only: the lanes beyond them repeat what lies 64 bytes before, and nobody reads it */
		const auto request = [&](int piece, auto slot) __attribute__((always_inline))
		{
			const int back = (piece * 128 + 64 == k_bytes) ? (chunk & 64) : 0;
#pragma unroll
			for (int u = 0; u < LOADS; u++)
			{
				__builtin_amdgcn_global_load_lds((global_ptr_t) (src[u] - back), (lds_ptr_t) (lds + decltype(slot)::value * Shape::SLOT_BYTES + (wave + WAVES * u) * 1024), 16, 0, 0);
				src[u] += 128;
			}
		};
		request(0, std::integral_constant<int, 0>());
		if (pieces > 1)
			request(1, std::integral_constant<int, 1>());

		acc_vec acc[BLOCKS_M][BLOCKS_N];
#pragma unroll
		for (int i = 0; i < BLOCKS_M; i++)
#pragma unroll
			for (int j = 0; j < BLOCKS_N; j++)
#pragma unroll
				for (int r = 0; r < 16; r++)
					acc[i][j][r] = 0;
		int a_first[BLOCKS_M], b_first[BLOCKS_N]; /* this lane's fragment of a slot's first k step, the others by XOR */
#pragma unroll
		for (int i = 0; i < BLOCKS_M; i++)
		{
			const int row = wave_m * 32 * BLOCKS_M + 32 * i + frag_row;
			a_first[i] = row * 128 + ((half_sel ^ ((row >> 1) & 7)) * 16);
		}
#pragma unroll
		for (int j = 0; j < BLOCKS_N; j++)
		{
			const int row = Shape::BM + wave_n * 32 * BLOCKS_N + 32 * j + frag_row;
			b_first[j] = row * 128 + ((half_sel ^ ((row >> 1) & 7)) * 16);
		}
		const auto multiply = [&](int piece, auto slot) __attribute__((always_inline))
		{
			/* loads return in order: this piece has landed once at most those of the next one are outstanding */
			if (piece + 1 < pieces)
				wait_vmcnt<LOADS>();
			else
				wait_vmcnt<0>();
			barrier_no_fence();
			const uint8_t *base = lds + decltype(slot)::value * Shape::SLOT_BYTES;
			const auto step = [&](int kk) __attribute__((always_inline))
			{
				uint4_t a[BLOCKS_M], b[BLOCKS_N];
#pragma unroll
				for (int i = 0; i < BLOCKS_M; i++)
					a[i] = *reinterpret_cast<const uint4_t*>(base + (a_first[i] ^ (kk * 32)));
#pragma unroll
				for (int j = 0; j < BLOCKS_N; j++)
					b[j] = *reinterpret_cast<const uint4_t*>(base + (b_first[j] ^ (kk * 32)));
#pragma unroll
				for (int i = 0; i < BLOCKS_M; i++)
#pragma unroll
					for (int j = 0; j < BLOCKS_N; j++)
						Traits::mma(b[j], a[i], acc[i][j]);
			};
			step(0);
			step(1);
			if (piece * 128 + 64 < k_bytes)
			{
				step(2);
				step(3);
			}
			/* everyone has read the slot before it takes the piece after the next one, or the slabs of the store */
			wait_lgkmcnt_zero();
			if (piece + 2 < pieces)
			{
				barrier_no_fence();
				request(piece + 2, slot);
			}
		};
		for (int piece = 0; piece < pieces; piece += 2)
		{
			multiply(piece, std::integral_constant<int, 0>());
			if (piece + 1 < pieces)
				multiply(piece + 1, std::integral_constant<int, 1>());
		}
		barrier_no_fence();

		/* lane l, register r of block (i, j): m = 32 i + l % 32, n = 32 j + 16 (l / 32) + r; 32 rows at a time cross the wavefront's slab and
		 * leave as whole rows of the sub-tile, 16 bytes per lane (N is a multiple of the vector, checked by the launcher) */
		constexpr int E = 16 / sizeof(T), LANES_PER_ROW = 32 * BLOCKS_N / E, ROWS_PER_PASS = 64 / LANES_PER_ROW;
		uint8_t *slab = lds + wave * 32 * Shape::SLAB_STRIDE;
		T *out = C + matrix * stride_c;
		const int col = (lane % LANES_PER_ROW) * E;
#pragma unroll
		for (int i = 0; i < BLOCKS_M; i++)
		{
#pragma unroll
			for (int j = 0; j < BLOCKS_N; j++)
#pragma unroll
				for (int r = 0; r < 16; r += E)
				{
					Vec<T, E> v;
#pragma unroll
					for (int e = 0; e < E; e++)
						v.v[e] = acc[i][j][r + e];
					v.store(reinterpret_cast<T*>(slab + frag_row * Shape::SLAB_STRIDE) + 32 * j + 16 * half_sel + r);
				}
			wait_lgkmcnt_zero(); /* the slab is private to this wavefront */
			__builtin_amdgcn_wave_barrier();
#pragma unroll
			for (int pass = 0; pass < 32 / ROWS_PER_PASS; pass++)
			{
				const int row = pass * ROWS_PER_PASS + lane / LANES_PER_ROW;
				const uint4_t v = *reinterpret_cast<const uint4_t*>(slab + row * Shape::SLAB_STRIDE + col * sizeof(T));
				const int m = m0 + 32 * i + row;
				if (m < M && n0 + col < N)
					*reinterpret_cast<uint4_t*>(out + static_cast<size_t>(m) * N + n0 + col) = v;
			}
			wait_lgkmcnt_zero();
			__builtin_amdgcn_wave_barrier();
		}
	}

	template<typename T, int BLOCKS_M, int BLOCKS_N, int WAVES_M, int WAVES_N>
	inline bool try_launch_gemm_tiles_as(hipStream_t stream, const StreamGemmArgs &g, bool by_rows)
	{
		typedef GemmTileShape<T, BLOCKS_M, BLOCKS_N, WAVES_M, WAVES_N> Shape;
		const int tiles_m = ceil_div(g.M, Shape::BM), tiles_n = ceil_div(g.N, Shape::BN);
		const unsigned long long tiles = static_cast<unsigned long long>(tiles_m) * tiles_n * g.batch;
		if (tiles > 0xffffffffULL / Shape::THREADS) /* threads that a launch can have */
			return false;
		auto kernel = kernel_gemm_tiles_nt<T, Shape>;
		if (Shape::LDS_BYTES > 64 * 1024)
			ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), Shape::LDS_BYTES);
		hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned int>(tiles)), dim3(Shape::THREADS), Shape::LDS_BYTES, stream, reinterpret_cast<const T*>(g.A),
				reinterpret_cast<const T*>(g.B), reinterpret_cast<T*>(g.C), g.M, g.N, g.k_bytes, g.stride_a, g.stride_b, g.stride_c, tiles_m, tiles_n, g.batch, by_rows);
		return true;
	}
	/* what the products read once and write: all of A and C */
	inline unsigned long long exchanged_bytes(const StreamGemmArgs &g, int element_size)
	{
		return static_cast<unsigned long long>(g.batch) * g.M * (static_cast<unsigned long long>(g.k_bytes) + static_cast<unsigned long long>(g.N) * element_size);
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
		return g.batch >= 8 && g.M >= 192 && exchanged_bytes(g, element_size) <= (40ULL << 20);
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
				|| (g.batch >= 8 && g.M >= 8 * static_cast<long long>(g.N) && 2 * b_bytes <= (5ULL << 20) && exchanged_bytes(g, element_size) <= (112ULL << 20));
	}
	/*
	 * Whether these tiles take a batch of plain products, by the number of 32x32 tiles and the bytes of A and C (figures as above, other
	 * kernel / this one).
	 * Not where the direct kernel's 32x32 tiles are few enough to be ahead: 256-byte rows, 128 channels, 448 rows (2016 tiles) 13.0 / 14.1 us, 512 (2304) 12.9 /
	 * 12.1; 512: 256 channels, 96 rows (864) 10.4 / 10.7, 128 (1152) 11.3 / 11.0; 384: 192 channels, 96 rows (648) 9.0 / 9.4, 160 (1080) 10.6 / 10.5; 768: 384
	 * channels, 32 rows (432) 10.5 / 11.2, 64 (864) 13.0 / 12.2; and fp32 rows of 384 bytes and more but 512, for which the small tiles of conv_tiles.hpp stand:
	 * 192 channels, 32 rows (216) 10.7 / 11.6, 64 (432) 13.8 / 12.2.
	 * Not beyond a number of bytes where the streaming kernel, which fetches A once, or for 64 and 128 bytes the kernels that store more at
	 * a time are level or ahead: fp16 256-byte rows 57 MB 32.2 / 28.8, 75 35.3 / 33.7, but with three calls per layer 23.6 / 24.0 and 94 MB 28.3 / 29.5; 512: 94 MB 53.3 / 53.3, 113 59.1 / 61.4, 302 127 / 143; 768, of
	 * which the streaming kernel holds only 128 columns: 226 MB 132 / 120, with three calls per layer 280 MB 150 / 160; fp32 512-byte rows 151 MB 82.4 / 79.9, 227
	 * 117 / 123; 64-byte rows (the stem, alone) 170 MB 32.4 / 29.3, 340 89.8 / 101; fp32 128-byte rows 85 MB 25.3 / 26.2, 149 31.0 / 33.6, 255 49.1 / 65.0.
	 */
	inline bool gemm_tiles_apply(const StreamGemmArgs &g, int element_size)
	{
		const bool fp16 = element_size == 2;
		if (g.k_bytes % 64 != 0 || (fp16 && (g.k_bytes == 128 || g.k_bytes > 768)))
			return false;
		const long long tiles = static_cast<long long>(ceil_div(g.M, 32)) * ceil_div(g.N, 32) * g.batch;
		long long fewest = 0; /* 32x32 tiles per compute unit */
		unsigned long long megabytes = ~0ULL >> 20; /* most of A and C together */
		switch (g.k_bytes)
		{
			case 64:
				megabytes = 270;
				break;
			case 128:
				megabytes = 100;
				break;
			case 256:
				fewest = fp16 ? 8 : 0;
				megabytes = fp16 ? 64 : megabytes;
				break;
			case 384:
				fewest = fp16 ? 4 : 1;
				break;
			case 512:
				fewest = fp16 ? 4 : 0;
				megabytes = fp16 ? 90 : 200;
				break;
			case 768:
				fewest = fp16 ? 3 : 1;
				megabytes = fp16 ? 220 : megabytes;
				break;
			default:
				fewest = (fp16 || g.k_bytes < 384) ? 0 : 1;
				break;
		}
		return tiles >= fewest * device_compute_units() && exchanged_bytes(g, element_size) <= (megabytes << 20);
	}
	/*
	 * Larger tiles, which fetch less, once there are enough of them. fp16 by rows, 64x64 / 128x64: 256 channels 448 rows (1008 tiles of 64x64) 18.6 / 19.2, 512
	 * (1152) 19.8 / 19.1; 128 channels 896... 960 rows (1080) 16.1 / 16.0; 384 channels 192 rows (648) 18.9 / 19.4, 256 (864) 21.6 / 20.6. By matrix, 128x64 / 128x128:
	 * 192 channels 2304 rows 32.8 / 35.5; 256 channels 1616 rows 37.8 / 36.7, 2304 52.2 / 51.2; 384 channels 1408 rows 58.4 / 55.1, 3072 97.5 / 95.6. fp32 stays at
	 * 64x64: 128 channels 2048 rows 45.6 / 46.0, 256 channels 960 63.0 / 65.5, 640 46.7 / 45.8 (128x64).
	 */
	template<typename T>
	inline bool try_launch_gemm_tiles(hipStream_t stream, const StreamGemmArgs &g)
	{
		if (!gemm_tiles_apply(g, sizeof(T)))
			return false;
		const bool by_rows = products_go_by_rows(g, sizeof(T));
		if constexpr (sizeof(T) == 2)
		{
			const long long tiles = static_cast<long long>(ceil_div(g.M, 64)) * ceil_div(g.N, 64) * g.batch;
			if (tiles >= (g.k_bytes >= 768 ? 3 : 4) * device_compute_units())
			{
				if (!by_rows && g.k_bytes >= 512)
					return try_launch_gemm_tiles_as<T, 2, 1, 2, 4>(stream, g, false);
				return try_launch_gemm_tiles_as<T, 2, 1, 2, 2>(stream, g, by_rows);
			}
		}
		return try_launch_gemm_tiles_as<T, 1, 1, 2, 2>(stream, g, by_rows);
	}
} /* namespace mlhip */

#endif /* MINML_AMD_GEMM_TILES_HPP_ */
