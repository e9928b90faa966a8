# ab.sh <name> <cases> [extra]
bash /root/repo/_work/p/g.sh $1 600 "timeout -k 10 560 python3 _work/arch_task/perf.py ab --start _work/start --only $2 $3" 40
